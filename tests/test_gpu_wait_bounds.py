"""Waits inside kernels end at a bound: a pair's workgroup then makes its chain
alone, and a streamed answer is packed and chained again before its stream
goes on."""
import ctypes as C

import numpy as np
import pytest

import inspire_amd as ia
import oracle_lib as ol
from oracle_lib import N

pytestmark = pytest.mark.gpu
SEED = np.array([0x42] + [0] * 63, np.uint8)
NQ = 35  # a sub-batch of 32 and one of 3


@pytest.fixture(scope="module")
def table():
    n, w, rows = 524288, 120, 2048
    rc, geo = ol.setup(n, w, rows)
    assert rc == 0
    db = np.random.default_rng(8).integers(0, ol.P, size=(geo["R"], geo["C"]), dtype=np.uint16)
    srv = ia.Server(db, n, w, rows, max_batch=NQ, crs_seed=bytes(SEED))
    lib = srv.lib
    qs = [ol.make_query(geo, SEED, 1000 * k + 5, 70 + k)[0] for k in range(NQ)]
    assert lib.ipir_dbg_set_group_chunk(srv.h, 2) == 0
    assert lib.ipir_dbg_set_pipeline(srv.h, 0, 0) == 0
    assert lib.ipir_dbg_set_horner(srv.h, 0) == 0
    want = srv.answer_batch(qs)
    assert lib.ipir_dbg_set_horner(srv.h, -1) == 0
    yield geo, srv, qs, want
    srv.close()


@pytest.mark.parametrize("shape", [0, 2, 3, 6, 7, 8])
@pytest.mark.parametrize("limit", [1, 6])
def test_answers_past_their_wait_bounds(table, shape, limit):
    """Bounds of a few loads, which streamed packs and chains always exceed
    and pairs now and then: right on every entry point, nothing reported."""
    geo, srv, qs, want = table
    lib, words = srv.lib, geo["T"] * 4 * N
    assert lib.ipir_dbg_set_pipeline(srv.h, shape, shape) == 0
    for cls in (1, NQ):
        assert lib.ipir_dbg_set_stream_slices(srv.h, cls, 4) == 0
    assert lib.ipir_dbg_set_horner_spin_limit(srv.h, limit) == 0
    assert lib.ipir_dbg_set_stream_spin_limit(srv.h, limit) == 0
    lib.ipir_dbg_chains_redone(srv.h)
    n0 = lib.ipir_dbg_streamed_count(srv.h)
    cl = ia.Client(srv.params, lib)
    try:
        for first, nq in ((0, 3), (2, 1), (0, NQ), (7, 16)):
            part, ref = qs[first: first + nq], want[first: first + nq]
            out = np.zeros_like(ref)
            assert lib.ipir_answer_batch(srv.h, srv.views(part), nq, ia.ptr(out)) == 0, nq
            assert np.array_equal(out, ref), nq
            dq, dout = ia.DeviceBuffer(nq * part[0].nbytes, lib), ia.DeviceBuffer(ref.nbytes, lib)
            dq.upload(np.stack(part))
            assert lib.ipir_answer_batch_device(srv.h, C.c_void_p(dq.p), nq, C.c_void_p(dout.p), None) == 0
            assert lib.ipir_device_status(srv.h) == 0
            assert np.array_equal(dout.download(np.zeros_like(ref)), ref), f"device, {nq}"
            comp = srv.answer_packed(np.stack([cl.pack_query(q) for q in part]))
            assert np.array_equal(comp, np.stack([cl.compress(r) for r in ref])), f"packed, {nq}"
            dq.free()
            dout.free()
        loop = lib.ipir_loop_start(srv.h, 2)
        assert loop
        try:
            got = np.zeros((4, words), np.uint64)
            tickets = [lib.ipir_loop_submit(loop, srv.views([qs[k]]), ia.ptr(got[k])) for k in range(4)]
            assert [lib.ipir_loop_wait(loop, t, None) for t in tickets] == [0] * 4
            assert np.array_equal(got, want[:4])
        finally:
            lib.ipir_loop_stop(loop)
        redone = lib.ipir_dbg_chains_redone(srv.h)
        print(f"[bounds] shape {shape} limit {limit}: redone {redone}")
        if lib.ipir_dbg_streamed_count(srv.h) != n0:
            assert redone == 1, "streamed chains wait longer than a few loads"
        assert lib.ipir_dbg_chains_redone(srv.h) == 0
    finally:
        assert lib.ipir_dbg_set_horner_spin_limit(srv.h, 1 << 21) == 0
        assert lib.ipir_dbg_set_stream_spin_limit(srv.h, 1 << 23) == 0
    out = np.zeros_like(want[:3])
    assert lib.ipir_answer_batch(srv.h, srv.views(qs[:3]), 3, ia.ptr(out)) == 0
    assert np.array_equal(out, want[:3])
    assert lib.ipir_dbg_chains_redone(srv.h) == 0, "ordinary bounds are not reached"


def test_pair_bound_is_at_most_the_default(table):
    """A bound past the default (2^26 was it, in another unit) is the default:
    no pair holds its CUs for minutes."""
    _, srv, _, _ = table
    lib = srv.lib
    default = lib.ipir_dbg_horner_spin_limit(srv.h)
    assert default == 1 << 21
    for limit, got in ((0, 0), (7, 7), (1 << 26, default), (1 << 21, default), ((1 << 32) - 1, default)):
        assert lib.ipir_dbg_set_horner_spin_limit(srv.h, limit) == 0
        assert lib.ipir_dbg_horner_spin_limit(srv.h) == got, limit
