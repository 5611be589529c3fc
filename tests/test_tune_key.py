"""The autotuner's stored choices: one counts for the kernels and the precision it was timed on, and for no others (CPU)."""

import json
import shutil

import pytest
import torch

from maxichem_amd import _kernels, _tables, standin, tune


@pytest.fixture
def store(tmp_path, monkeypatch):
    monkeypatch.setattr(tune, "STORE", tmp_path / "tune.json")
    monkeypatch.setattr(torch.cuda, "get_device_name", lambda device=None: "device")
    net = standin.load("NCHO")
    for mixed in (False, True):  # unlike the stored choice below
        assert tune.default_variant(_tables.build(net, True), mixed) != (1, 8, 1, 0)

    def put(key: str) -> None:
        tune.STORE.write_text(json.dumps({key: {"best": [1, 8, 1, 0]}}))

    return net, put


def test_a_choice_counts_for_its_kernels_only(store, tmp_path, monkeypatch):
    net, put = store
    put(tune._key(net, True, "cuda"))
    assert tune.choose(net, "cuda", True, 1e-6) == (1, 8, 1, 0)
    other = tmp_path / "kernels"
    shutil.copytree(_kernels.KERNEL_DIR, other)
    (other / "recover.hip").write_text((other / "recover.hip").read_text() + "// another kernel\n")
    monkeypatch.setattr(_kernels, "KERNEL_DIR", other)
    assert tune.choose(net, "cuda", True, 1e-6) == tune.default_variant(_tables.build(net, True))


def test_a_choice_without_its_kernels_does_not_count(store):
    net, put = store
    put(f"{_tables.build(net, True).digest()}|1|device")  # as stored before choices named their kernels
    assert tune.choose(net, "cuda", True, 1e-6) == tune.default_variant(_tables.build(net, True))


def test_the_mixed_form_takes_only_its_own_choice(store):
    net, put = store
    put(tune._key(net, True, "cuda"))
    assert tune.choose(net, "cuda", True, 1e-6, mixed=True) == tune.default_variant(_tables.build(net, True), True)
    put(tune._key(net, True, "cuda", mixed=True))
    assert tune.choose(net, "cuda", True, 1e-6, mixed=True) == (1, 8, 1, 0)
    assert tune.choose(net, "cuda", True, 1e-6) == tune.default_variant(_tables.build(net, True))
