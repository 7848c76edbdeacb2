"""Chunked answers of several response ciphertexts, whose chains run on one
or two streams: two ciphertexts whose chunks end with them, and three whose
chunks straddle two (768 groups in chunks of 96), equal to the serial answers
and extracting to their entries."""
import numpy as np
import pytest

import inspire_amd as ia
import oracle_lib as ol

pytestmark = pytest.mark.gpu
SEED = np.array([0x42] + [0] * 63, np.uint8)


@pytest.mark.parametrize("cts", [2, 3])
def test_chunked_answers_of_several_ciphertexts(cts):
    n, w, rows, nq = cts << 24, 120, 2048, 3
    rc, geo = ol.setup(n, w, rows)
    assert rc == 0 and geo["G"] == 256 * cts and geo["T"] == cts
    part = np.random.default_rng(cts).integers(0, ol.P, size=(geo["R"] // 8, geo["C"]), dtype=np.uint16)
    db = np.tile(part, (8, 1))
    srv = ia.Server(db, n, w, rows, max_batch=nq, crs_seed=bytes(SEED))
    lib = srv.lib
    try:
        idx = [5, n // 2 + 77, n - 1]
        qs, sts = zip(*[ol.make_query(geo, SEED, i, 60 + k) for k, i in enumerate(idx)])
        assert lib.ipir_dbg_set_horner(srv.h, 0) == 0
        assert lib.ipir_dbg_set_pipeline(srv.h, 0, 0) == 0
        want = srv.answer_batch(list(qs))
        for k, i in enumerate(idx):
            got = ol.extract(geo, sts[k], want[k].reshape(geo["T"], -1))
            assert np.array_equal(got, ol.expected_slots(geo, db, i)), f"entry {i}"
        for shape in (2, 3, 4):
            assert lib.ipir_dbg_set_pipeline(srv.h, shape, shape) == 0
            for split in (0, 1, 3):
                assert lib.ipir_dbg_set_tail_split(srv.h, split) == 0
                for mode in (0, -1):
                    assert lib.ipir_dbg_set_horner(srv.h, mode) == 0
                    print(f"[{cts} cts] shape {shape} split {split} horner {mode}", flush=True)
                    for order in ([0, 1, 2], [2, 0, 1], [1]):  # other queries in the same slots
                        got = srv.answer_batch([qs[j] for j in order])
                        assert np.array_equal(got, want[order]), (shape, split, mode, order)
        # pairs that do not wait for their partner: each workgroup makes its chain alone
        assert lib.ipir_dbg_set_horner_spin_limit(srv.h, 1) == 0
        for shape in (0, 2, 3):
            assert lib.ipir_dbg_set_pipeline(srv.h, shape, shape) == 0
            print(f"[{cts} cts] shape {shape}, bound of one load", flush=True)
            assert np.array_equal(srv.answer_batch(list(qs)), want), f"alone, shape {shape}"
    finally:
        srv.close()
