"""Kernels at the edges of their ranges against the oracle: the largest
residues through the unfolded transforms of the Horner chain."""
import numpy as np
import pytest

import inspire_amd as ia
import oracle_lib as ol
from oracle_lib import BLK, N

pytestmark = pytest.mark.gpu
Q = np.array([ol.Q0, ol.Q1], np.uint64)


def _polys(kind, shape, seed):
    """RNS polynomials [..., limb, N] of extreme values: every residue q-1,
    alternating 0 and q-1, or q-1 in the first slot of each 8 only."""
    x = np.zeros(shape + (2, N), np.uint64)
    if kind == "largest":
        x += (Q - 1)[:, None]
    elif kind == "alternating":
        x[..., ::2] = (Q - 1)[:, None]
    elif kind == "sparse":
        x[..., ::8] = (Q - 1)[:, None]
    else:
        x = ol.rand_poly(np.random.default_rng(seed), shape)
    return np.ascontiguousarray(x)


@pytest.mark.parametrize("rgsw", ["largest", "alternating", "random"])
@pytest.mark.parametrize("cts", ["largest", "alternating", "sparse", "random"])
def test_horner_chain_of_extreme_residues(cts, rgsw):
    L = 4
    c = _polys(cts, (L, 2), 1).reshape(-1)
    r = _polys(rgsw, (4, 2), 2).reshape(-1)
    assert r.size == 4 * BLK
    out, want = np.zeros(4 * N, np.uint64), np.zeros(4 * N, np.uint64)
    assert ia.load("server").ipir_dbg_horner(ia.ptr(c), L, ia.ptr(r), ia.ptr(out)) == 0
    ol.oracle().orc_horner(c, L, r, want)
    assert np.array_equal(out, want)
