"""The device's sets of streams for pipelined answers, put together while other
threads keep the device busy: each set's streams run side by side."""
import threading

import numpy as np
import pytest
import torch

import inspire_amd as ia
import oracle_lib as ol

pytestmark = pytest.mark.gpu
SEED = np.array([0x42] + [0] * 63, np.uint8)


@pytest.mark.parametrize("threads", [0, 4, 8])
def test_sets_made_on_a_busy_device(threads):
    n, w, rows = 262144, 120, 2048
    rc, geo = ol.setup(n, w, rows)
    db = np.random.default_rng(8).integers(0, ol.P, size=(geo["R"], geo["C"]), dtype=np.uint16)
    e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    torch.cuda._sleep(1000000)
    e0.record()
    torch.cuda._sleep(1000000)
    e1.record()
    e1.synchronize()
    cycles = int(1000000 * 0.5 / e0.elapsed_time(e1))  # half a millisecond
    stop = threading.Event()

    def load():
        stream = torch.cuda.Stream()
        while not stop.is_set():
            with torch.cuda.stream(stream):
                for _ in range(4):
                    torch.cuda._sleep(cycles)
            stream.synchronize()

    ts = [threading.Thread(target=load) for _ in range(threads)]
    for t in ts:
        t.start()
    srv = None
    try:
        srv = ia.Server(db, n, w, rows, max_batch=2, crs_seed=bytes(SEED))
    finally:
        stop.set()
        for t in ts:
            t.join()
    torch.cuda.synchronize()
    try:
        assert srv.lib.ipir_dbg_lanes_apart(srv.h) == 4
    finally:
        srv.close()
