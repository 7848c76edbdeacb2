"""Answers inside a caller's own stream capture: the first one a server gives
in its pipelined shapes, captured in global mode (in which no thread may
create what the capture would depend on), replayed over other queries."""
import ctypes as C

import numpy as np
import pytest
import torch

import inspire_amd as ia
import oracle_lib as ol
from oracle_lib import N

pytestmark = pytest.mark.gpu
SEED = np.array([0x42] + [0] * 63, np.uint8)
NQ = 3


@pytest.mark.parametrize("shape", [0, 2, 3, 6])
def test_first_answer_of_a_shape_in_a_callers_capture(shape):
    n, w, rows = 524288, 120, 2048
    rc, geo = ol.setup(n, w, rows)
    db = np.random.default_rng(8).integers(0, ol.P, size=(geo["R"], geo["C"]), dtype=np.uint16)
    srv = ia.Server(db, n, w, rows, max_batch=2 * NQ, crs_seed=bytes(SEED))
    lib = srv.lib
    try:
        qs = [ol.make_query(geo, SEED, 1000 * k + 5, 70 + k)[0] for k in range(2 * NQ)]
        assert lib.ipir_dbg_set_group_chunk(srv.h, 2) == 0
        assert lib.ipir_dbg_set_pipeline(srv.h, 0, 0) == 0
        want = srv.answer_batch(qs)
        assert lib.ipir_dbg_set_pipeline(srv.h, shape, shape) == 0
        dq = torch.zeros(NQ * qs[0].size, dtype=torch.int64, device="cuda")
        out = torch.zeros((NQ, geo["T"] * 4 * N), dtype=torch.int64, device="cuda")
        stream, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
        torch.cuda.synchronize()
        with torch.cuda.graph(graph, stream=stream, capture_error_mode="global"):
            rc = lib.ipir_answer_batch_device(srv.h, C.c_void_p(dq.data_ptr()), NQ, C.c_void_p(out.data_ptr()),
                                              C.c_void_p(stream.cuda_stream))
        assert rc == 0
        for rep in range(4):
            first = rep % 2 * NQ
            dq.copy_(torch.from_numpy(np.concatenate(qs[first: first + NQ]).view(np.int64)))
            out.fill_(-1)
            graph.replay()
            torch.cuda.synchronize()
            got = out.cpu().numpy().view(np.uint64)
            assert np.array_equal(got, want[first: first + NQ]), f"replay {rep}"
            assert np.array_equal(srv.answer_batch(qs), want), "eager work between the replays"
        assert lib.ipir_device_status(srv.h) == 0
    finally:
        srv.close()
