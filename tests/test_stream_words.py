"""The kernels' stream words: each carries its entry's destination, and adding the terms one by one at those places
gives the sums of the tables' entries (CPU)."""

import numpy as np
import pytest

from maxichem_amd import _kernels, _tables, standin
from maxichem_amd._tables import SV_DBL, SV_END, SV_PIECE, SV_R_BITS, T_DBL, T_DEST, T_END, T_IDX_BITS


def sums(words, values, idx_bits, dbl, dest, size):
    """What the kernels' stream adds: each word's term at its destination, a lane's words in order."""
    out = np.zeros(size)
    for lane in range(words.shape[1]):
        for w in words[:, lane]:
            w = int(w)
            d = values[w & ((1 << idx_bits) - 1)] * (2.0 if w >> dbl & 1 else 1.0) * (-1.0 if w >> 31 else 1.0)
            out[(w & 0x7FFFFFFF) >> dest] += d
    return out


def entries(words, values, idx_bits, dbl, end, dest, size):
    """The tables' own meaning: a running sum per lane, stored where a word ends an entry."""
    out = np.zeros(size)
    for lane in range(words.shape[1]):
        acc = 0.0
        for w in words[:, lane]:
            w = int(w)
            acc += values[w & ((1 << idx_bits) - 1)] * (2.0 if w >> dbl & 1 else 1.0) * (-1.0 if w >> 31 else 1.0)
            if w >> end & 1:
                out[(w & 0x7FFFFFFF) >> dest] = acc
                acc = 0.0
    return out


@pytest.mark.parametrize("stem", ["synthetic", "synthetic_small", "synthetic_decay", "NCHO", "SNCHO"])
def test_every_word_goes_to_its_entry(read_network, stem):
    tab = _tables.build(standin.load(stem) if stem.endswith("NCHO") else read_network(stem), True)
    host = _kernels.host_tables(tab)
    rng = np.random.default_rng(0)
    size = tab.layout()["SIZE"]
    dv = np.append(rng.standard_normal(tab.ndv), 0.0)  # dv[ndv] = 0: the padding words' term
    for mine, kernel in ((tab.diag_words, "diagw"), (tab.lead_words, "leadw"), (np.concatenate(tab.chunk_words), "chw")):
        w = host[kernel].view(np.uint32).reshape(mine.shape)
        assert np.array_equal(w & 0x3FFFF | w & 0x80000000, mine & 0x3FFFF | mine & 0x80000000)
        if kernel == "chw":  # one chunk at a time: the chunks share their destinations
            rounds = np.cumsum([0] + [c.shape[0] for c in tab.chunk_words])
            parts = [(w[a:b], mine[a:b]) for a, b in zip(rounds, rounds[1:])]
        else:
            parts = [(w, mine)]
        for got, want in parts:
            assert np.array_equal(sums(got, dv, T_IDX_BITS, T_DBL, T_DEST, size),
                                  entries(want, dv, T_IDX_BITS, T_DBL, T_END, T_DEST, size))  # fmt: skip
    v = np.append(rng.standard_normal(tab.nr), 0.0)
    w = host["svw"].view(np.uint32).reshape(tab.sv_words.shape)
    assert np.array_equal(sums(w, v, SV_R_BITS, SV_DBL, SV_PIECE, tab.npart),
                          entries(tab.sv_words, v, SV_R_BITS, SV_DBL, SV_END, SV_PIECE, tab.npart))  # fmt: skip
