"""The stream words' destinations: word by word what a lane's own list of entries says, also where a lane ends no entry;
and a solver's construction does not wait for them (CPU)."""

import time

import numpy as np
import pytest

from maxichem_amd import _kernels, _tables, standin

END, DEST = 16, 18


def one_lane(words, spare):
    """A lane's words with the destination of the entry each belongs to: its next ended one, else its last, else spare."""
    ends = [i for i, w in enumerate(words) if w >> END & 1]
    out = []
    for i, w in enumerate(words):
        owner = next((e for e in ends if e >= i), ends[-1] if ends else None)
        place = int(spare) if owner is None else (words[owner] & 0x7FFFFFFF) >> DEST
        out.append((w & ~(0x1FFF << DEST)) | place << DEST)
    return out


@pytest.mark.parametrize("rounds", [1, 2, 7, 33])
@pytest.mark.parametrize("share", [0.0, 0.2, 1.0])
def test_every_word_has_its_entrys_destination(rounds, share):
    rng = np.random.default_rng(rounds)
    words = rng.integers(0, 2**32, (rounds, 64), dtype=np.uint64).astype(np.uint32) & ~np.uint32(1 << END)
    words |= (rng.random((rounds, 64)) < share).astype(np.uint32) << np.uint32(END)
    spare = rng.integers(0, 2**13, 64)
    got = _kernels.every_destination(words, END, DEST, spare)
    assert got.dtype == np.uint32
    assert got.T.tolist() == [one_lane([int(w) for w in words[:, q]], spare[q]) for q in range(64)]


@pytest.mark.parametrize("shape", ["NCHO", "SNCHO"])
def test_the_words_cost_little_beside_the_tables(shape):
    net = standin.load(shape)

    def best(f):
        took = []
        for _ in range(5):
            start = time.perf_counter()
            f()
            took.append(time.perf_counter() - start)
        return min(took)

    tab = _tables.build(net, True)
    assert best(lambda: _kernels.host_tables(tab)) < best(lambda: _tables.build(net, True)) / 12.0
