"""A reaction whose efficiency is below 0 (the reader takes every finite one, and a solver any rate table): its rates and
its derivatives are negative, and the Jacobian takes them with their sign (GPU)."""

import numpy as np
import oracle
import pytest
from test_kernel_pieces import probe

from maxichem_amd import standin

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("stem", ["synthetic", "NCHO"])
def test_the_jacobian_takes_negative_rates_with_their_sign(read_network, stem):
    net = standin.load(stem) if stem == "NCHO" else read_network(stem)
    turned = [r for r in net.reac if "eff" in r]
    for r in turned:
        r["eff"] = -r["eff"]
    assert turned
    x = 10.0 ** np.random.default_rng(4).uniform(-8, 0, len(net.species))
    x /= x.sum()
    T, P = 1700.0, 3e5
    tab, got = probe(net, False, x, T, P, 1e-4, None)
    kf, kr = oracle.Oracle(tab).rates(T, P)
    assert kf.min() < 0.0 and kr.min() < 0.0
    F, JN = oracle.Oracle(tab).rhs_jacobian(T, P, x)
    # as for the positive rates: sums of a few terms, each rounded
    np.testing.assert_allclose(got["F"], F, rtol=1e-10, atol=1e-12 * np.abs(F).max())
    np.testing.assert_allclose(got["w"][:, None] - got["mjn"], JN, rtol=1e-9, atol=1e-12 * np.abs(JN).max())
