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


SEED = np.array([0x42] + [0] * 63, np.uint8)
# rows that are no power of two (ranges of 4096 rows end in a half one), one
# group (the pack writes the responses) and two (chains of two ciphertexts)
ODD = {"one group": (40000, 120, 10240), "two groups": (300000, 59, 6144)}


@pytest.fixture(scope="module", params=sorted(ODD))
def odd_table(request):
    n, w, rows = ODD[request.param]
    rc, geo = ol.setup(n, w, rows)
    assert rc == 0
    db = np.random.default_rng(3).integers(0, ol.P, size=(geo["R"], geo["C"]), dtype=np.uint16)
    pc = ol.OraclePrecomp(db, geo, SEED)
    srv = ia.Server(db, n, w, rows, max_batch=33, crs_seed=bytes(SEED))
    qs = [ol.make_query(geo, SEED, (i * 7919) % n, 900 + i)[0] for i in range(33)]
    yield geo, pc, srv, qs, [None] * 33
    srv.close()


@pytest.mark.parametrize("nq", [1, 2, 3, 5, 9, 16, 17, 33])
def test_batches_of_every_pass_form_match_oracle(odd_table, nq):
    """Every form of the preparation launch (1..4 digit rows per limb, the
    7-digit rows, a sub-batch of one after 32), residues up to the prime and
    beyond it."""
    geo, pc, srv, qs, want = odd_table
    batch = [q.copy() for q in qs[:nq]]
    batch[-1][: geo["R"]] += np.uint64(ol.Q0)             # reduced on the way in
    batch[-1][geo["R"]: 2 * geo["R"]] += np.uint64(7 * ol.Q1)
    got = srv.answer_batch(batch)
    for i in range(nq):
        if want[i] is None:
            want[i] = pc.answer(qs[i]).reshape(-1)
        assert np.array_equal(got[i], want[i]), f"query {i} of {nq}"
