"""The timed database pass runs over the queries of the last call that staged
some, in whatever form that call left them."""
import ctypes as C

import numpy as np
import pytest

import inspire_amd as ia
import oracle_lib as ol
from oracle_lib import N

pytestmark = pytest.mark.gpu
SEED = np.array([0x42] + [0] * 63, np.uint8)


def test_timed_pass_takes_the_staged_queries():
    # two groups, 240 MB: blocking calls of 9 to 32 queries stage the LWE parts apart
    n, w, rows = 2 << 20, 120, 32768
    rc, geo = ol.setup(n, w, rows)
    assert rc == 0
    R, cols = geo["R"], geo["C"]
    db = np.random.default_rng(4).integers(0, ol.P, size=(R, cols), dtype=np.uint16)
    srv = ia.Server(db, n, w, rows, max_batch=16, crs_seed=bytes(SEED))
    lib = srv.lib
    try:
        assert lib.ipir_dbg_set_pipeline(srv.h, 0, 0) == 0
        qs = np.stack([ol.make_query(geo, SEED, 7919 * k, 40 + k)[0] for k in range(16)])
        ref = np.zeros((16, 2, cols), np.uint32)
        assert lib.ipir_dbg_db_pass(srv.h, ia.ptr(np.ascontiguousarray(qs[:, : 2 * R])), 16, -1, ia.ptr(ref)) == 0
        cl = ia.Client(srv.params, lib)
        dq, out = ia.DeviceBuffer(qs.nbytes, lib), ia.DeviceBuffer(16 * geo["T"] * 4 * N * 8, lib)
        stages = (C.c_double * 5)()

        def profile(order):
            dq.upload(np.ascontiguousarray(qs[order]))
            assert lib.ipir_dbg_profile_batch(srv.h, C.c_void_p(dq.p), len(order), C.c_void_p(out.p), stages) == 0

        def loop(order):
            lp = lib.ipir_loop_start(srv.h, 1)
            got = np.zeros(geo["T"] * 4 * N, np.uint64)
            ticket = lib.ipir_loop_submit(lp, srv.views([qs[order[0]]]), ia.ptr(got))
            assert lib.ipir_loop_wait(lp, ticket, None) == 0
            lib.ipir_loop_stop(lp)

        calls = {
            "blocking": lambda o: srv.answer_batch(list(qs[o])),
            "packed": lambda o: srv.answer_packed(np.stack([cl.pack_query(q) for q in qs[o]])),
            "profiled": profile,
            "loop": loop,
        }
        for name, call in calls.items():
            for order in ([3], [5, 1, 2], list(range(12, 2, -1))):
                if name == "loop":
                    order = order[:1]
                call(order)
                ms, got = C.c_double(), np.zeros((len(order), 2, cols), np.uint32)
                assert lib.ipir_dbg_time_dbpass(srv.h, len(order), 1, C.byref(ms)) == 0 and ms.value > 0
                assert lib.ipir_dbg_interm(srv.h, len(order), ia.ptr(got)) == 0
                assert np.array_equal(got, ref[order]), (name, order)
        dq.free()
        out.free()
    finally:
        srv.close()
