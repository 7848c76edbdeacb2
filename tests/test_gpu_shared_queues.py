"""Servers of one device share its hardware queues: a server's answers beside
those of another one whose caller's stream is busy for long."""
import ctypes as C
import threading

import numpy as np
import pytest
import torch

import inspire_amd as ia
import oracle_lib as ol
from oracle_lib import N

pytestmark = pytest.mark.gpu
SEED = np.array([0x42] + [0] * 63, np.uint8)
NQ = 3


class Device:
    """A flat batch on the device and room for its responses."""

    def __init__(self, lib, qs, resp_words):
        self.lib = lib
        self.q = ia.DeviceBuffer(qs.nbytes, lib)
        self.q.upload(qs)
        self.out = ia.DeviceBuffer(8 * resp_words * len(qs), lib)
        self.shape = (len(qs), resp_words)

    def answer(self, srv, stream):
        assert self.lib.ipir_answer_batch_device(srv.h, C.c_void_p(self.q.p), self.shape[0], C.c_void_p(self.out.p),
                                                 stream) == 0

    def get(self):
        return self.out.download(np.zeros(self.shape, np.uint64))


@pytest.fixture(scope="module")
def servers():
    """Six servers (more than the device has sets of streams) of one table."""
    n, w, rows = 524288, 120, 2048
    rc, geo = ol.setup(n, w, rows)
    assert rc == 0
    db = np.random.default_rng(8).integers(0, ol.P, size=(geo["R"], geo["C"]), dtype=np.uint16)
    srvs = [ia.Server(db, n, w, rows, max_batch=NQ, crs_seed=bytes(SEED)) for _ in range(6)]
    qs = np.stack([ol.make_query(geo, SEED, 1000 * k + 5, 70 + k)[0] for k in range(NQ)])
    lib = srvs[0].lib
    assert lib.ipir_dbg_set_pipeline(srvs[0].h, 0, 0) == 0
    want = srvs[0].answer_batch(list(qs))
    yield geo, lib, srvs, qs, want
    for s in srvs:
        s.close()


def busy_cycles(ms):
    """torch.cuda._sleep argument for about ms milliseconds (one workgroup)."""
    e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    torch.cuda._sleep(1000000)
    e0.record()
    torch.cuda._sleep(1000000)
    e1.record()
    e1.synchronize()
    return int(1000000 * ms / e0.elapsed_time(e1))


@pytest.mark.parametrize("shape", [6, 7, 8])
def test_streamed_answers_beside_busy_callers(servers, shape):
    """Server 0's streamed answers, their wait bound lowered to some 20 ms,
    beside another server's answers on a stream that is busy for 60 ms and on
    a second one, which the library makes wait for the first: that wait holds
    up a hardware queue (each of the device's in turn, over 8 streams), put
    there before server 0's answers and, from another thread, during them. It
    is never between server 0's waiting kernels and what they wait for, so no
    wait ends at its bound."""
    geo, lib, srvs, qs, want = servers
    words = geo["T"] * 4 * N
    cycles = busy_cycles(60)
    mine, theirs = Device(lib, qs, words), Device(lib, qs, words)
    a, b = srvs[0], srvs[1]
    assert lib.ipir_dbg_set_stream_slices(a.h, NQ, 4) == 0
    assert lib.ipir_dbg_set_pipeline(a.h, shape, shape) == 0
    assert lib.ipir_dbg_set_stream_spin_limit(a.h, 1 << 14) == 0
    assert lib.ipir_dbg_set_pipeline(b.h, 0, 0) == 0
    views = a.views(list(qs))
    out = np.zeros_like(want)
    busy = torch.cuda.Stream()
    streams = [lib.ipir_dev_stream_create() for _ in range(8)]
    lib.ipir_dbg_chains_redone(a.h)
    n0 = lib.ipir_dbg_streamed_count(a.h)
    try:
        for k, second in enumerate(streams):
            for beside in (False, True):
                print(f"[queues] shape {shape}, stream {k}, {'during' if beside else 'before'}", flush=True)
                failed = []

                def other():
                    try:
                        for _ in range(8 if beside else 1):
                            theirs.answer(b, C.c_void_p(busy.cuda_stream))
                            theirs.answer(b, second)
                    except Exception as e:  # noqa: BLE001 (reported below)
                        failed.append(e)

                with torch.cuda.stream(busy):
                    torch.cuda._sleep(cycles)
                t = threading.Thread(target=other)
                t.start()
                if not beside:
                    t.join()
                try:
                    for _ in range(8):
                        mine.answer(a, None)
                    assert lib.ipir_answer_batch(a.h, views, NQ, ia.ptr(out)) == 0
                finally:
                    t.join()
                assert not failed, failed
                assert lib.ipir_dev_sync() == 0
                assert np.array_equal(out, want)
                assert np.array_equal(mine.get(), want) and np.array_equal(theirs.get(), want)
                assert lib.ipir_dbg_chains_redone(a.h) == 0, f"a wait ended at its bound: stream {k}, {beside}"
        assert lib.ipir_dbg_streamed_count(a.h) - n0 == 8 * 2 * 9
    finally:
        assert lib.ipir_dev_sync() == 0
        assert lib.ipir_dbg_set_stream_spin_limit(a.h, 1 << 23) == 0
        for s in streams:
            lib.ipir_dev_stream_destroy(s)
