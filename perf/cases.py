"""The work that users of this library have it do, as measurable cases.

A case is a table (its geometry), how many queries are answered at once and
the entry point they go through:

  device  ipir_answer_batch_device: flat queries and responses resident in
          HBM, enqueued on the program's one stream (a service that moves
          queries itself, or answers what another kernel produced)
  host    ipir_answer_batch: the blocking C ABI call over host buffers, what
          a service that links this library in the reference's place calls
  packed  ipir_answer_batch_packed: the blocking call over packed wire
          queries and compressed responses, as they cross the network
  create  ipir_server_create, one answer and ipir_server_destroy: a new
          database generation, from the host's rows to its first response

Every output is a residue or a wire byte, exact integers that do not depend
on the order of the arithmetic.
"""
import concurrent.futures
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "inspire-gpu_amd"))
import inspire_amd as ia  # noqa: E402

N = ia.N
PLAIN = 65535            # database values are in [0, 2^16 - 1)
RESIDUE_BITS = 27        # of one resident tensor entry
SLOT_STEPS = 2046        # collapse entries per slot and digit
HALF_NTT = 11 * N // 2   # butterflies of one 2048-point transform


def listed():
    return [
        # the smallest table setup() takes (one 2048-row group), one lookup through
        # the C ABI: launches, copies and waits, hardly any memory traffic
        {"name": "tiny host x1", "entry": "host", "n_entries": 256, "entry_bytes": 120, "db_rows": 2048,
         "max_batch": 4, "batch": 1},
        # 0.13 GB, 2^20 x 60 B: a single latency-bound lookup, and a full batch
        {"name": "0.13GB x1", "entry": "device", "n_entries": 1 << 20, "entry_bytes": 60, "db_rows": 32768,
         "max_batch": 32, "batch": 1},
        {"name": "0.13GB x32", "entry": "device", "n_entries": 1 << 20, "entry_bytes": 60, "db_rows": 32768,
         "max_batch": 32, "batch": 32},
        # 1 GB, 2^23 x 120 B: the ordinary table, at one query, at a full batch, and
        # as a service calls it: flat host buffers, and a ragged batch off the wire
        {"name": "1GB x1", "entry": "device", "n_entries": 1 << 23, "entry_bytes": 120, "db_rows": 32768,
         "max_batch": 32, "batch": 1},
        {"name": "1GB x32", "entry": "device", "n_entries": 1 << 23, "entry_bytes": 120, "db_rows": 32768,
         "max_batch": 32, "batch": 32},
        {"name": "1GB host x32", "entry": "host", "n_entries": 1 << 23, "entry_bytes": 120, "db_rows": 32768,
         "max_batch": 32, "batch": 32},
        {"name": "1GB packed x13", "entry": "packed", "n_entries": 8000001, "entry_bytes": 119, "db_rows": 32768,
         "max_batch": 16, "batch": 13},
        # 4 GB of wide records (2^20 x 3840 B), a handful of queries at once
        {"name": "4GB wide x6", "entry": "device", "n_entries": 1 << 20, "entry_bytes": 3840, "db_rows": 32768,
         "max_batch": 8, "batch": 6},
        # 512 groups, so two ciphertexts per response as in the largest tables, at the
        # shortest query (2048 rows): the collapse and long Horner chains dominate
        {"name": "two cts x3", "entry": "device", "n_entries": 1 << 25, "entry_bytes": 120, "db_rows": 2048,
         "max_batch": 8, "batch": 3},
        # 16 GB, 2^27 x 120 B: the benchmark's table, one query and a full batch
        {"name": "16GB x1", "entry": "device", "n_entries": 1 << 27, "entry_bytes": 120, "db_rows": 32768,
         "max_batch": 32, "batch": 1},
        {"name": "16GB x32", "entry": "device", "n_entries": 1 << 27, "entry_bytes": 120, "db_rows": 32768,
         "max_batch": 32, "batch": 32},
        # a 1 GB table is replaced: upload, encode, precomputation, setup, first answer
        {"name": "1GB create", "entry": "create", "n_entries": 1 << 23, "entry_bytes": 120, "db_rows": 32768,
         "max_batch": 32, "batch": 1},
    ]


def draw(rng):
    """A table of 2048 to 32768 rows and 1 to 128 groups (8 MB to 16 GB), any entry
    width setup() takes, 1 to 48 queries at once through any entry point."""
    entry = rng.choice(["device", "device", "device", "host", "packed", "create"])
    groups = 1 << rng.randint(0, 4 if entry == "create" else 7)
    rows = 2048 * max(1, min(16, round(2 ** rng.uniform(0, 4))))
    chunks = 1 << rng.randint(0, 11)                     # 15-bit values per entry
    entry_bytes = max(1, chunks * 15 // 8)
    if entry_bytes > 1 and -(-(entry_bytes - 1) * 8 // 15) == chunks and rng.random() < 0.5:
        entry_bytes -= 1
    full = groups * N * rows // chunks
    n_entries = max(1, full - rng.randint(0, max(1, N // 2 * rows // chunks)))
    most = 48 if groups * rows <= 1 << 20 else 32        # no more work than the largest listed case
    batch = max(1, min(most, round(2 ** rng.uniform(0, 5.6))))
    if entry == "create":
        batch = 1
    max_batch = max(batch, 1 << rng.randint(0, 5))
    return {"entry": entry, "n_entries": n_entries, "entry_bytes": entry_bytes, "db_rows": rows,
            "max_batch": max_batch, "batch": batch}


def _geometry(case):
    return ia.geometry(case["n_entries"], case["entry_bytes"], case["db_rows"])


def _database(geo, seed):
    """Uniform values, rows generated on host threads."""
    rows, cols = geo["R"], geo["C"]
    db = np.empty((rows, cols), np.uint16)
    step = max(1, (1 << 25) // cols)
    starts = list(range(0, rows, step))
    seeds = np.random.SeedSequence(seed).spawn(len(starts))

    def fill(k):
        part = db[starts[k]:starts[k] + step]
        part[:] = np.random.default_rng(seeds[k]).integers(0, PLAIN, size=part.shape, dtype=np.uint16)
    with concurrent.futures.ThreadPoolExecutor(min(16, os.cpu_count() or 1)) as pool:
        list(pool.map(fill, range(len(starts))))
    return db


_program_stream = None


def _stream():
    """The one stream the program enqueues its device calls on."""
    global _program_stream
    if _program_stream is None:
        _program_stream = torch.cuda.Stream()
    return _program_stream.cuda_stream


def prepare(case, seed):
    geo = _geometry(case)
    rng = np.random.default_rng(seed)
    crs_seed = rng.integers(0, 256, 64, dtype=np.uint8).tobytes()
    db = _database(geo, seed)
    state = {"case": case, "lib": ia.load("server")}
    if case["entry"] == "create":
        params = ia.make_params(case["n_entries"], case["entry_bytes"], case["db_rows"], crs_seed, geo["R"], geo["C"],
                                geo["G"], geo["D"], geo["T"])
        state.update(db=db, crs_seed=crs_seed)
    else:
        srv = ia.Server(db, case["n_entries"], case["entry_bytes"], case["db_rows"], max_batch=case["max_batch"],
                        crs_seed=crs_seed)
        params = srv.params
        state["srv"] = srv
    client = ia.Client(params, state["lib"])
    queries = []
    for k in range(case["batch"]):
        secret, query = client.build(int(rng.integers(0, case["n_entries"])), int(rng.integers(0, 1 << 62)))
        client.destroy(secret)
        queries.append(query)
    count, cts = case["batch"], geo["T"]
    if case["entry"] == "device":
        state["queries"] = torch.from_numpy(np.stack(queries).view(np.int64)).cuda()
        state["responses"] = torch.empty((count, cts * 4 * N), dtype=torch.int64, device="cuda")
        state["stream"] = _stream()
    elif case["entry"] == "packed":
        state["queries"] = np.stack([client.pack_query(q) for q in queries])
        state["responses"] = np.zeros((count, cts * 12288), np.uint8)
    else:
        state["queries"] = queries
        state["responses"] = np.zeros((count, cts * 4 * N), np.int64)
        if case["entry"] == "host":
            state["views"] = state["srv"].views(queries)
    return state


def run(state):
    case, lib, out = state["case"], state["lib"], state["responses"]
    if case["entry"] == "device":
        rc = lib.ipir_answer_batch_device(state["srv"].h, state["queries"].data_ptr(), case["batch"], out.data_ptr(),
                                          state["stream"])
    elif case["entry"] == "host":
        rc = lib.ipir_answer_batch(state["srv"].h, state["views"], case["batch"], ia.ptr(out))
    elif case["entry"] == "packed":
        rc = lib.ipir_answer_batch_packed(state["srv"].h, ia.ptr(state["queries"]), case["batch"], ia.ptr(out))
    else:
        srv = ia.Server(state["db"], case["n_entries"], case["entry_bytes"], case["db_rows"],
                        max_batch=case["max_batch"], crs_seed=state["crs_seed"])
        rc = lib.ipir_answer_batch(srv.h, srv.views(state["queries"]), 1, ia.ptr(out))
        srv.close()
    if rc:
        raise RuntimeError("answer failed: %d" % rc)
    return out


def work(case):
    """Each table and tensor read once, each query read and response written once;
    two operations for a multiply-accumulate, three for a transform's butterfly."""
    geo = _geometry(case)
    rows, cols, groups, cts, count = geo["R"], geo["C"], geo["G"], geo["T"], case["batch"]
    table = 2 * rows * cols
    tensors = groups * 2 * 2 * SLOT_STEPS * N * RESIDUE_BITS // 8
    if case["entry"] == "packed":
        wire = count * ((rows + 12 * N) * 53 // 8 + cts * 12288)
    else:
        wire = count * 8 * (2 * rows + 24 * N + cts * 4 * N)
    steps = groups - cts  # external products of one query's chains
    flops = count * (4 * rows * cols + 4 * groups * 2 * SLOT_STEPS * N
                     + 3 * HALF_NTT * (12 * steps + 2 * groups + 8) + steps * 32 * N)
    moved = table + tensors + wire
    if case["entry"] == "create":
        moved += 2 * table + tensors  # the encoded table is written too, and the tensors once
        depth = max(1, min(256, groups))
        flops += (table // 2 * depth.bit_length()                   # encode
                  + 3 * HALF_NTT * 2 * (cols * rows // N + groups * N)  # a-side, ring embedding
                  + groups * 2 * (SLOT_STEPS // 2) * 6 * 3 * HALF_NTT)  # collapse chains
    return {"bytes": float(moved), "flops": float(flops)}


def exact(case, seed):
    """None: outputs are residues and wire bytes, whole numbers that have to be equal."""
    return None
