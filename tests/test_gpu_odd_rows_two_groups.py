"""Answers over a table of two groups whose rows are no power of two, so that
a row range of the preparation launch and of a pass's slices ends in a part:
every batch form, each response equal to the oracle's, with chains of two
groups as pairs and as one workgroup."""
import numpy as np
import pytest

import inspire_amd as ia
import oracle_lib as ol

pytestmark = pytest.mark.gpu
SEED = np.array([0x42] + [0] * 63, np.uint8)


def test_two_groups_of_odd_rows_match_the_oracle():
    n, w, rows = 393216, 120, 6144
    rc, geo = ol.setup(n, w, rows)
    assert rc == 0 and geo["G"] == 2 and geo["T"] == 1
    db = np.random.default_rng(3).integers(0, ol.P, size=(geo["R"], geo["C"]), dtype=np.uint16)
    pc = ol.OraclePrecomp(db, geo, SEED)
    srv = ia.Server(db, n, w, rows, max_batch=33, crs_seed=bytes(SEED))
    try:
        qs = [ol.make_query(geo, SEED, (i * 7919) % n, 900 + i)[0] for i in range(33)]
        want = np.stack([pc.answer(q).reshape(-1) for q in qs])
        for mode in (-1, 0):
            assert srv.lib.ipir_dbg_set_horner(srv.h, mode) == 0
            for nq in (1, 2, 3, 5, 9, 16, 17, 33):
                assert np.array_equal(srv.answer_batch(qs[:nq]), want[:nq]), (mode, nq)
    finally:
        srv.close()
