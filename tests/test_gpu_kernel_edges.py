"""Kernels at the edges of their ranges against the oracle: the largest
residues through the unfolded transforms of the Horner chain."""
import ctypes as C

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


def test_servers_on_one_device_stream_side_by_side():
    """Six servers share the device's four sets of streams for pipelined
    answers: streamed answers enqueued back to back on two streams without
    waiting equal the serial one."""
    n, w, rows, nq = 524288, 120, 2048, 3
    rc, geo = ol.setup(n, w, rows)
    db = np.random.default_rng(8).integers(0, ol.P, size=(geo["R"], geo["C"]), dtype=np.uint16)
    lib = ia.load("server")
    srvs = [ia.Server(db, n, w, rows, max_batch=nq, crs_seed=bytes(SEED)) for _ in range(6)]
    streams = [lib.ipir_dev_stream_create() for _ in range(2)]
    qs = np.stack([ol.make_query(geo, SEED, 1000 * k + 5, 70 + k)[0] for k in range(nq)])
    dq = ia.DeviceBuffer(qs.nbytes, lib)
    dq.upload(qs)
    outs = [ia.DeviceBuffer(nq * geo["T"] * 4 * N * 8, lib) for _ in srvs]
    try:
        for s in srvs:
            assert lib.ipir_dbg_stream_ok(s.h) == 1
            assert lib.ipir_dbg_set_pipeline(s.h, 0, 0) == 0
        want = srvs[0].answer_batch(list(qs))
        for s in srvs:
            assert lib.ipir_dbg_set_stream_slices(s.h, nq, 4) == 0
            assert lib.ipir_dbg_set_pipeline(s.h, 6, 6) == 0
        before = [lib.ipir_dbg_streamed_count(s.h) for s in srvs]
        for s in srvs:
            assert np.array_equal(s.answer_batch(list(qs)), want)
        assert [lib.ipir_dbg_streamed_count(s.h) - b for s, b in zip(srvs, before)] == [1] * 6
        for rnd in range(4):
            for k, s in enumerate(srvs):
                assert lib.ipir_answer_batch_device(s.h, C.c_void_p(dq.p), nq, C.c_void_p(outs[k].p),
                                                    streams[k % 2]) == 0
        assert lib.ipir_dev_sync() == 0
        for k, s in enumerate(srvs):
            assert lib.ipir_device_status(s.h) == 0
            assert np.array_equal(outs[k].download(np.zeros_like(want)), want), f"server {k}"
    finally:
        for s in srvs:
            s.close()
        for st in streams:
            lib.ipir_dev_stream_destroy(st)


def test_wire_words_beyond_32_bits_and_unaligned_packed_buffers(odd_table):
    """Residues plus large multiples of their prime, over 2^32, through the
    narrowing host entry and the 64-bit device entry; packed queries and
    compressed responses at odd device addresses."""
    geo, pc, srv, qs, want = odd_table
    lib, R, nq = srv.lib, geo["R"], 5
    base = srv.answer_batch(qs[:nq])
    wide = np.stack([q.copy() for q in qs[:nq]])
    rng = np.random.default_rng(12)
    limb = np.concatenate([np.zeros(R, int), np.ones(R, int), np.tile(np.repeat([0, 1], N), 12)])
    k = rng.integers(0, 1 << 36, wide.shape, dtype=np.uint64)
    k[:, ::3] = 0  # some words stay canonical
    wide += k * Q[limb][None, :]
    assert wide.max() > 1 << 60
    assert np.array_equal(srv.answer_batch(list(wide)), base)
    dq, dout = ia.DeviceBuffer(wide.nbytes, lib), ia.DeviceBuffer(base.nbytes, lib)
    dq.upload(wide)
    assert lib.ipir_answer_batch_device(srv.h, C.c_void_p(dq.p), nq, C.c_void_p(dout.p), None) == 0
    assert lib.ipir_dev_sync() == 0
    assert np.array_equal(dout.download(np.zeros_like(base)), base)
    cl = ia.Client(srv.params, lib)
    packed = np.stack([cl.pack_query(q) for q in qs[:nq]])
    comp = srv.answer_packed(packed)
    assert np.array_equal(comp, np.stack([cl.compress(r) for r in base]))
    for off in (1, 8, 16):
        src = np.concatenate([np.zeros(off, np.uint8), packed.reshape(-1)])
        dp, dc = ia.DeviceBuffer(src.nbytes, lib), ia.DeviceBuffer(comp.nbytes + off, lib)
        dp.upload(src)
        assert lib.ipir_answer_batch_packed_device(srv.h, C.c_void_p(dp.p + off), nq, C.c_void_p(dc.p + off), None) == 0
        assert lib.ipir_dev_sync() == 0
        assert np.array_equal(dc.download(np.zeros(comp.nbytes + off, np.uint8))[off:], comp.reshape(-1)), off


@pytest.mark.parametrize("rgsw", ["largest", "alternating", "random"])
@pytest.mark.parametrize("cts", ["largest", "alternating", "sparse", "random"])
def test_pair_chain_of_extreme_residues(cts, rgsw):
    """The same chain by a workgroup pair, whose teams add two products."""
    L = 4
    c = _polys(cts, (L, 2), 1).reshape(-1)
    r = _polys(rgsw, (4, 2), 2).reshape(-1)
    out, want = np.zeros(4 * N, np.uint64), np.zeros(4 * N, np.uint64)
    assert ia.load("server").ipir_dbg_horner_variant(ia.ptr(c), L, ia.ptr(r), ia.ptr(out), 1) == 0
    ol.oracle().orc_horner(c, L, r, want)
    assert np.array_equal(out, want)


def test_pair_chain_longer_than_its_step_numbers():
    """1030 steps: the exchange's numbers 1..1023 start again."""
    L = 1031
    c = _polys("random", (L, 2), 5).reshape(-1)
    r = _polys("random", (4, 2), 6).reshape(-1)
    out, want = np.zeros(4 * N, np.uint64), np.zeros(4 * N, np.uint64)
    assert ia.load("server").ipir_dbg_horner_variant(ia.ptr(c), L, ia.ptr(r), ia.ptr(out), 1) == 0
    ol.oracle().orc_horner(c, L, r, want)
    assert np.array_equal(out, want)


@pytest.mark.parametrize("shape", [0, 2])
def test_pair_chains_of_plain_answers(shape):
    """Answers whose chains run as pairs by themselves, in one launch and in
    one per chunk: equal to the one-workgroup kernel's, on blocking and
    device calls; a wait over its bound (0: every kernel still ends) is
    reported and leaves no residue in the response, and the next answer is
    right again."""
    n, w, rows, nq = 524288, 120, 2048, 3
    rc, geo = ol.setup(n, w, rows)
    db = np.random.default_rng(8).integers(0, ol.P, size=(geo["R"], geo["C"]), dtype=np.uint16)
    lib = ia.load("server")
    srv = ia.Server(db, n, w, rows, max_batch=nq, crs_seed=bytes(SEED))
    qs = np.stack([ol.make_query(geo, SEED, 1000 * k + 5, 70 + k)[0] for k in range(nq)])
    dq = ia.DeviceBuffer(qs.nbytes, lib)
    dq.upload(qs)
    out = ia.DeviceBuffer(nq * geo["T"] * 4 * N * 8, lib)

    def device():
        assert lib.ipir_answer_batch_device(srv.h, C.c_void_p(dq.p), nq, C.c_void_p(out.p), None) == 0
        assert lib.ipir_dev_sync() == 0
        return out.download(np.zeros_like(want))

    try:
        assert lib.ipir_dbg_set_group_chunk(srv.h, 2) == 0
        assert lib.ipir_dbg_set_pipeline(srv.h, shape, shape) == 0
        assert lib.ipir_dbg_set_horner(srv.h, 0) == 0
        want = srv.answer_batch(list(qs))
        assert lib.ipir_dbg_set_horner(srv.h, -1) == 0
        for _ in range(3):
            assert np.array_equal(srv.answer_batch(list(qs)), want)
            assert np.array_equal(device(), want)
        assert lib.ipir_dbg_set_horner_spin_limit(srv.h, 0) == 0
        assert (device() == ~np.uint64(0)).all()
        assert lib.ipir_device_status(srv.h) == 4
        assert lib.ipir_answer_batch(srv.h, srv.views(list(qs)), nq, ia.ptr(np.zeros_like(want))) == 4
        assert lib.ipir_dbg_set_horner_spin_limit(srv.h, 1 << 21) == 0
        assert np.array_equal(device(), want)
        assert lib.ipir_device_status(srv.h) == 0
    finally:
        out.free()
        dq.free()
        srv.close()


@pytest.mark.parametrize("groups,shape", [(1, 0), (2, 0), (2, 3)])
def test_staged_batches_whose_keys_follow_the_pass(groups, shape):
    """Host and packed calls of 8 to 33 queries over 128 and 240 MB (from 9
    to 32 and two groups on, serial, the keys and RGSW rows reach the device
    beside the pass), a different set of queries each call: equal to the
    device entry's answers."""
    n, w, rows = groups << 20, 120 if groups > 1 else 60, 32768
    rc, geo = ol.setup(n, w, rows)
    assert rc == 0 and geo["G"] == groups
    db = np.random.default_rng(4).integers(0, ol.P, size=(geo["R"], geo["C"]), dtype=np.uint16)
    lib = ia.load("server")
    srv = ia.Server(db, n, w, rows, max_batch=33, crs_seed=bytes(SEED))
    try:
        assert lib.ipir_dbg_set_pipeline(srv.h, shape, shape) == 0
        qs = np.stack([ol.make_query(geo, SEED, 7919 * k, 40 + k)[0] for k in range(33)])
        dq = ia.DeviceBuffer(qs.nbytes, lib)
        dq.upload(qs)
        out = ia.DeviceBuffer(33 * geo["T"] * 4 * N * 8, lib)
        assert lib.ipir_answer_batch_device(srv.h, C.c_void_p(dq.p), 33, C.c_void_p(out.p), None) == 0
        assert lib.ipir_dev_sync() == 0
        want = out.download(np.zeros((33, geo["T"] * 4 * N), np.uint64))
        cl = ia.Client(srv.params, lib)
        packed = np.stack([cl.pack_query(q) for q in qs])
        comp = np.stack([cl.compress(r) for r in want])
        for first, nq in ((0, 8), (3, 9), (20, 13), (1, 32), (0, 33), (11, 10)):
            part = slice(first, first + nq)
            assert np.array_equal(srv.answer_batch(list(qs[part])), want[part]), (first, nq)
            assert np.array_equal(srv.answer_packed(packed[part]), comp[part]), (first, nq)
        dq.free()
        out.free()
    finally:
        srv.close()


@pytest.mark.parametrize("groups,rows", [(2, 2048), (4, 2048), (16, 2048), (32, 2048), (64, 2048), (1, 34 * 2048)])
def test_preprocessing_of_every_group_count_extracts(groups, rows):
    """The encode's power-of-two extents (2..64 groups of interpolation
    points) and a-side sums of 1 and of 34 polynomials (past the 32 between
    reductions): first, middle and last entry extract."""
    n, w = groups * rows * N // 64, 120
    rc, geo = ol.setup(n, w, rows)
    assert rc == 0 and geo["G"] == groups
    db = np.random.default_rng(groups).integers(0, ol.P, size=(geo["R"], geo["C"]), dtype=np.uint16)
    srv = ia.Server(db, n, w, rows, max_batch=1, crs_seed=bytes(SEED))
    try:
        for k, idx in enumerate((0, n // 2 + 1, n - 1)):
            q, st = ol.make_query(geo, SEED, idx, 50 + k)
            got = ol.extract(geo, st, srv.answer_batch([q])[0].reshape(geo["T"], -1))
            assert np.array_equal(got, ol.expected_slots(geo, db, idx)), f"entry {idx}"
    finally:
        srv.close()
