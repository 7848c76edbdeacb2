// Internal definition of the opaque GpuServerCtx (not installed).
#pragma once
#include <hip/hip_runtime.h>

#include <functional>
#include <atomic>
#include <mutex>
#include <utility>
#include <vector>

#include "capi.h"
#include "chunks.h"
#include "gpu_protocol.h"
#include "host_stage.h"
#include "kernels.h"
#include "lanes.h"

namespace inspire {

void hip_check(hipError_t e, const char* what);
inline void dfree(void* p) {
    if (p) (void)hipFree(p);
}

// The key and RGSW parts of staged queries that reach the device beside the
// database pass, which needs the LWE parts alone.
struct LateKeys {
    std::function<void(hipStream_t)> copy;  // to the device, on the side stream (waits for the host job)
    std::function<void(hipStream_t)> after; // what is left to do behind the copy, on the answer's stream
    const uint32_t* words = nullptr;        // then: stride words per query, the key part first
    size_t stride = 0;
};

// Flat queries an answer starts from: u64 wire words, or words narrowed to
// u32 (back to back, qlen words each), in device or pinned host memory; with
// `stage`, queries that a host job is still writing (query 0 is its item 0).
// With `late` (one sub-batch) the LWE parts alone, lwe_stride words apart.
struct QueryInput {
    const void* q = nullptr;
    bool narrow = false;
    HostStage* stage = nullptr;
    size_t first = 0;  // item of query 0
    const LateKeys* late = nullptr;
    size_t lwe_stride = 0;
    QueryInput(const uint64_t* d) : q(d) {}
    QueryInput(const uint32_t* d, HostStage* st = nullptr) : q(d), narrow(true), stage(st) {}
    QueryInput at(size_t k, size_t qlen) const {
        QueryInput x = *this;
        x.q = static_cast<const char*>(q) + k * qlen * (narrow ? 4 : 8);
        x.first += k;
        return x;
    }
};

struct GpuServerCtx {
    PublicParams pp{};
    GpuServerConfig cfg{};
    int device = 0;
    hipStream_t stream = nullptr;
    size_t G = 0, Da = 0, T = 0;

    // resident data
    // encoded DB, byte planes in 16-row blocks: plane p (low/high byte) of
    // (r, c) at byte ((r/16)*2 + p)*C*16 + c*16 + r%16
    uint16_t* d_db = nullptr;
    const uint8_t* db_planes() const { return reinterpret_cast<const uint8_t*>(d_db); }
    uint32_t* d_precomp = nullptr;  // [G][PC_GROUP] arena
    uint32_t* d_tw = nullptr;       // twiddles
    ipx::NttConst nc{};
    ipx::CrtConst cc{};

    // per-query slot pools, max_batch each
    ipx::SlotLayout lay{};
    ipx::DbPlan plan1{};            // database pass of a single query over all columns (autotuned)
    size_t plan1_target = 2048;     // its workgroup target
    size_t mfma_target = 1024;      // workgroups the batched pass aims for
    uint32_t mfma_depth = 4;        // register-ring depth of the 9..32-query passes
    int mfma_form = 0;              // 9..32 queries: form of the pass (dbplan_form)
    // 9..16 queries when timed apart from a larger largest batch (their
    // best form differs): target, depth and form
    bool tuned16 = false;
    size_t mfma16_target = 1024;
    uint32_t mfma16_depth = 4;
    int mfma16_form = 0;
    // row slices of the batched chunk plan, timed at setup for plans with
    // chunk_param digit tiles (0: the narrowing rule)
    uint32_t chunk_slices = 0, chunk_param = 0;
    // row slices of serial answers' full-width pass where timed below the
    // plan's (0: the plan's); of many-query answers for plans with
    // serial_param digit tiles
    uint32_t serial_slices = 0, serial_param = 0, serial_slices1 = 0;
    uint32_t chunk_slices1 = 0;     // the same for one-query answers (plan1's kind)
    // chunks from index late_from on (the collapse beside them has finished)
    // take late_slices row slices instead (0: as the chunks before them);
    // one-query answers use the *1 pair
    uint32_t late_from = 0, late_slices = 0, late_from1 = 0, late_slices1 = 0;
    // The plan of a chunk of ng groups at index k of the pipelined answer.
    ipx::DbPlan chunk_plan_at(size_t nq, size_t k, size_t ng, const ipx::DbPlan& whole) const;
    int collapse_variant = 0;       // 17..32-query collapse pass form (launch_collapse)
    size_t gchunk = 0;              // groups per chunk of the pipelined answer
    // the pipelined answer's chunks: of gchunk groups, the lowest one split
    // into gchunk/2, /4, /4 when tail_split (its Horner steps are the ones
    // left after every pass), the highest one into gchunk/4, /4, /2 when
    // head_split (the chains start after a quarter chunk's passes)
    bool tail_split = true, head_split = false;
    ChunkLayout layout;
    void set_chunks();
    // pipeline shape of one-query and many-query calls: 0 serial on the
    // caller's stream, 2 Horner chains beside the passes, 3 collapse beside
    // too, 4 the collapse of all groups before the database-pass chunks, 5
    // collapse beside and a chunk ahead; streamed (one full-width database
    // pass handing groups over as it runs, the chains waiting for them in
    // the kernel): 6 after the collapse of all groups, 7 with the collapse
    // beside, 8 with the collapse in the pass's own launch, group by group
    // (up to 8 queries) (2, 3, 6 and 8 timed at setup)
    int pipe_single = 3, pipe_batched = 2;
    int pipe_single_chunked = 3, pipe_batched_chunked = 3;  // where a streamed shape cannot run
    bool pipe_forced = false;       // INSPIRE_PIPELINE set the shapes (not autotuned)
    // row slices of the streamed pass (one query, many), and whether this
    // server may stream at all (INSPIRE_STREAM). The workgroups of a streamed
    // answer hold their CUs while they wait; the device's lane sets are
    // shared by its servers and run one answer's chains at a time each, so
    // at most kLanes answers wait, whatever servers they belong to. What they
    // wait for follows their release in its queue (lanes.h, QueueTurn).
    uint32_t stream_slices1 = 4, stream_slices = 4;
    // eighths of the groups (from the top) in a streamed pass's first
    // launch, the chains starting after it (0: one launch, chains at once)
    uint32_t stream_split1 = 0, stream_split = 0;
    bool stream_ok = false;
    // The streamed pass's plan for nq queries (the tuned kernel, the streamed
    // slice count, at least the slices exactness needs); kind F64 if none fits.
    // One- and two-query passes stream with 128-column tiles per wave (fewer,
    // longer workgroups per group), except inside the collapse's launch
    // (fused: the 64-column tiles its work items share).
    ipx::DbPlan stream_plan(size_t nq, uint32_t slices, bool fused = false) const;
    // Whether an answer on s may take a streamed shape now (not under capture).
    bool can_stream(hipStream_t s) const;
    // A streamed sub-batch of nq queries holds nq*T chain workgroups and
    // ceil(nq/pack_width(nq)) pack workgroups (one CU each) while they wait:
    // at most kStreamMaxWaiters, so 4 lanes leave 64 of 256 CUs to passes.
    static constexpr size_t kStreamMaxWaiters = 48;
    bool stream_fits(size_t nq) const;
    // Queries per streamed pack workgroup: 2 up to 16 queries (one round of
    // its 4 teams per group, so the pack keeps pace with the faster passes
    // of small batches), kPackQueries above (two rounds, fewer CUs held
    // beside the slower 17..32-query pass).
    static uint32_t pack_width(size_t nq) { return nq <= 16 ? 2u : ipx::kPackQueries; }
    size_t qlen = 0, resp_u64s = 0;
    size_t part_stride = 0, part2_stride = 0, keys_stride = 0, rgsw_stride = 0, packed_stride = 0;
    uint64_t* d_q = nullptr;        // flat queries (device staging)
    uint64_t* d_resp = nullptr;     // flat responses (device staging)
    double* d_bq = nullptr;
    uint32_t* d_keys = nullptr;
    uint32_t* d_rgsw = nullptr;
    uint32_t* d_part = nullptr;     // DB-pass row-slice partials [B][S][2][C]
    uint32_t* d_interm = nullptr;   // DB-pass result [B][2][C]
    uint32_t* d_part2 = nullptr;    // collapse sums [B][G][2][N]
    // scratch of the batched database pass, one set per concurrent lane
    static constexpr int kLanes = 4;
    int8_t* d_dig[kLanes] = {};     // query digits [R/16][<=256][16]
    uint32_t* d_S[kLanes] = {};     // digit-offset corrections [32][2][kOffsetSumParts]
    static constexpr size_t kSumWords = ipx::kMfmaMaxQueries * 2 * ipx::kOffsetSumParts;
    static constexpr size_t kKeySumWords = ipx::kCollapseMaxQueries * 2 * ipx::kKeySumParts;
    // scratch of the collapse pass: key digits [2][2N/16][<=128][16], key sums
    static constexpr size_t kKdigBytes = 2 * (2 * ipx::N / 16) * 128 * 16;
    int8_t* d_kdig[kLanes] = {};
    uint32_t* d_KS[kLanes] = {};
    // per lane, one set per 32-query sub-batch of a call: the streamed
    // pass's per-group completion counts [G], then the streamed pack's
    // per-(workgroup, group) publication flags [32 / kPackQueries][G]
    // (pack_width gives at most that many workgroups: 16 queries at 2)
    static constexpr size_t kStreamSetWords = 1 + ipx::kMfmaMaxQueries / ipx::kPackQueries;
    static_assert(16 / 2 <= ipx::kMfmaMaxQueries / ipx::kPackQueries, "pack workgroups of a 16-query sub-batch");
    uint32_t* d_sflags[kLanes] = {};
    size_t stream_sets = 0;
    // Per lane, the streams of pipelined answers: the database passes, and
    // beside them the Horner chains and the collapse or pack (lanes.h), with
    // the events that hand each group chunk over. A caller's stream may share
    // a hardware queue with either side stream, so pipelined answers hop from
    // it to the passes' stream and back.
    static constexpr int kChunkEvents = 16;
    LaneStreams lanes[kLanes];
    int lane_first = -1;  // acquire_lanes' answer
    hipStream_t capture_horner = nullptr, capture_side = nullptr;  // the side streams of captured answers
    hipEvent_t hop_in_ev[kLanes] = {}, hop_out_ev[kLanes] = {};
    hipEvent_t chunk_ev[kLanes][kChunkEvents] = {};  // database pass of a chunk done
    hipEvent_t coll_ev[kLanes][kChunkEvents] = {};   // collapse of a chunk done
    hipEvent_t prep_ev[kLanes] = {};                 // keys of a batch in place
    hipEvent_t pass_ev[kLanes] = {};                 // a split streamed pass's first launch done
    hipEvent_t horner_done[kLanes] = {};
    uint32_t* d_packed_b = nullptr;
    // Horner kernel of chains that do not wait for a streamed pass: -1 = a
    // workgroup pair per chain (one per limb) for up to kPairMaxChains of an
    // answer, else one workgroup; 0 = one workgroup always; 1 = pairs
    // always, except where nobody reads the call's status
    int horner_mode = -1;
    // pack kernel of pipelined chunks: 1 one workgroup per query, 0 a grid
    // over (group, limb), -1 one workgroup for one-query calls, 2 fused into
    // the Horner chains' own workgroups (where the one-workgroup Horner runs)
    int pack_wg = 0;
    uint32_t* d_hxbuf = nullptr;    // pair exchange buffers [B*T chains]
    // Waits inside a kernel (a pair chain's for its partner, a streamed pack's
    // or chain's for its pass) are bounded. A pair's workgroup whose wait ends
    // at its bound makes the chain alone (kernels_horner.hip). Streamed: per
    // scratch lane, d_gave_up is zeroed by an answer's first kernel and set by
    // such a wait, and the answer's last launches make its streamed
    // sub-batches again, without waits, where it is set. Both then set
    // h_status[kLanes] (pinned host memory). With a bound of zero (chains
    // that end at once, for tests) nothing is made again, the report goes to
    // h_status[lane], and check_status reads and clears it.
    uint32_t* d_gave_up = nullptr;  // [kLanes]
    uint32_t* h_status = nullptr;   // [kLanes + 1]
    uint32_t horner_spin_limit = 0; // the pair kernel's wait bound in loads (0: report at once)
    uint32_t stream_spin_limit = 0; // the same for chains waiting for a streamed pass's groups
    uint32_t* d_hstate = nullptr;   // Horner chain state between chunk launches [B*T][4][N]
    // Pinned host staging, which kernels read and write directly: queries
    // narrowed to u32 words (qlen per slot), or packed ones; flat or
    // compressed responses.
    uint32_t* h_q = nullptr;
    uint64_t* h_resp = nullptr;
    std::unique_ptr<HostStage> host_stage;  // fills h_q and empties h_resp
    static constexpr size_t kStageHelpers = 3;
    static constexpr size_t kStagePiece = 4;  // queries per preparation launch while the rest is staged
    // late_keys: from this many queries over a table of this size (bytes; a
    // pass of 20 us). Host calls of 3, 6, 9, 32 queries with everything before
    // the pass and with the late part: 240 MB 166 / 180, 215 / 229, 295 / 246,
    // 603 / 523 us; 1 GB 377 / 384, 417 / 408, 520 / 483, 887 / 794.
    static constexpr size_t kLateQueries = 9, kLateTableBytes = (size_t)1 << 27;
    static constexpr size_t kLatePiece = 8;   // queries per copy
    size_t lwe_packed_bytes() const { return pp.db_rows / 8 * 53; }  // of a packed query
    uint32_t* flat32() const { return reinterpret_cast<uint32_t*>(d_q); }  // unpacked queries

    // packed-wire path (53-bit CRT-packed queries in, compressed responses out)
    static constexpr size_t kCompressedCtBytes = ipx::N * (28 + 20) / 8;  // 12288
    size_t qpack_bytes = 0;
    uint32_t* d_cmp = nullptr;      // coefficient-form responses [B*T][4][N]

    size_t resident_bytes = 0;
    // mu serialises every entry point that touches the slots, scratch lanes
    // or plans; loop_active (under mu) marks a serving loop that owns them
    // until it stops, and those entry points then return "busy".
    std::mutex mu;
    bool loop_active = false;
    // Calls on lane 0 and slots [0, count) from different streams are
    // ordered: each waits for the previous one's work (order_ev, recorded on
    // order_stream) before enqueueing its own.
    hipEvent_t order_ev = nullptr;
    hipStream_t order_stream = nullptr;
    bool order_stream_set = false;
    void order_before(hipStream_t s);
    void order_after(hipStream_t s);
    // s waits for e, in a queue turn: every wait this library puts on a
    // stream goes through here (lanes.h, QueueTurn).
    void stream_wait(hipStream_t s, hipEvent_t e);

    // Captured answer steps: with graph_mode on, the first answer of a given
    // (input, output, count, slots, lane, form) is captured from its stream
    // into a hipGraph and every later one replays it. Kernel arguments are
    // frozen at capture, so anything that changes a plan drops the cache.
    struct StepGraph {
        const void* in;
        void* out;
        size_t count, slot0;
        int lane, packed;
        hipGraphExec_t exec;
    };
    static constexpr size_t kMaxGraphs = 64;
    int graph_mode = 0;
    std::vector<StepGraph> graphs;
    std::mutex graph_mu;  // the cache (device-side calls take no other lock)
    // fn enqueues the step on s; captured or replayed as above, run as is when
    // graph_mode is off or s is the null stream or already capturing.
    void run_step(const void* in, void* out, size_t count, size_t slot0, int lane, int packed, hipStream_t s,
                  const std::function<void()>& fn);
    void drop_graphs();

    void alloc_slots();
    // Pick the fastest database-pass variant on this device and geometry.
    void autotune_dbpass();
    // Pipeline stages over slots [q0, q0+nq) (one sub-batch, at most 32) on
    // stream s, their int8 operands in scratch set `lane`.
    // What an answer's first launch zeroes beside its own work.
    struct PrepZero {
        uint32_t* flags = nullptr;  // flag_words words
        uint32_t flag_words = 0;
        bool part2 = false;         // the collapse sums (a split collapse adds into them)
        bool pair = false;          // the pair chains' exchange words
        bool skip_lwe = false;      // leave the LWE part to prep_lwe
        uint32_t* status = nullptr, *gave_up = nullptr;  // a word each
    };
    ipx::PrepArgs prep_args(const QueryInput& in, size_t stride, size_t q0, int lane) const;
    // Keys, RGSW rows and plan p's pass operands of the flat queries at d_in.
    void prep_query(const QueryInput& in, size_t q0, size_t nq, const ipx::DbPlan& p, hipStream_t s, int lane,
                    const PrepZero& z);
    void prep_query(const QueryInput& in, size_t q0, size_t nq, const ipx::DbPlan& p, hipStream_t s, int lane) {
        prep_query(in, q0, nq, p, s, lane, PrepZero{});
    }
    // Plan p's pass operands alone, of LWE parts stride words apart (staged
    // ones piece by piece).
    void prep_lwe(const QueryInput& in, size_t stride, size_t q0, size_t nq, const ipx::DbPlan& p, hipStream_t s,
                  int lane);
    void launch_pieces(const ipx::PrepArgs& a, const QueryInput& in, size_t nq, const ipx::DbPlan& p, hipStream_t s);
    // Where a full-width pass of plan p writes: its row slices' partials, or interm.
    uint32_t* pass_out(size_t q0, const ipx::DbPlan& p, size_t& qstride);
    void dbpass_whole(size_t q0, size_t nq, const ipx::DbPlan& p, hipStream_t s, int lane);
    void collapse_whole(size_t q0, size_t nq, hipStream_t s, int lane, bool zeroed = false);
    // d_out: also the responses (tables of one group)
    void pack_whole(size_t q0, size_t nq, const ipx::DbPlan& p, hipStream_t s, uint64_t* d_out = nullptr);
    // The serial answer's plan: plan_for's at the timed row slices.
    ipx::DbPlan serial_plan(size_t nq) const;
    // The tuned database-pass plan for nq queries over ncols columns.
    ipx::DbPlan plan_for(size_t nq, size_t ncols) const;
    // The tuned full-width plan narrowed to ncols columns at its workgroup count.
    ipx::DbPlan chunk_plan(size_t nq, size_t ncols) const;
    // Database pass of queries [q0, q0+nq) over the columns of groups [g_lo, g_hi) into interm.
    void dbpass_range(size_t q0, size_t nq, size_t g_lo, size_t g_hi, const ipx::DbPlan& p, hipStream_t s, int lane);
    // Whether an answer's chains (of count queries) run as workgroup pairs.
    // Where set by hand, only where the caller reads the lane's status after
    // the call (status_read).
    bool use_pair(size_t count, bool status_read) const;
    // Horner chains of `count` queries over groups [g_lo, g_hi).
    // fp: the chains compute their groups' packed b-parts themselves first
    void horner_range(size_t count, uint64_t* d_out, size_t g_lo, size_t g_hi, hipStream_t s, size_t slot0,
                      int lane, bool pair, const ipx::FusedPack* fp = nullptr);
    // The chains of `count` queries in one launch and without waits, where a
    // streamed wait of the lane's answer ended at its bound.
    void horner_again(size_t count, uint64_t* d_out, hipStream_t s, size_t slot0, int lane);
    // Throw (and clear) if a chain of a call on `lane` gave up its wait with a
    // bound of zero (h_status); the call's stream has been waited for.
    void check_status(int lane);
    std::atomic<size_t> n_streamed{0};  // streamed sub-batches enqueued (a test counter)
    // row slices whose partials the last answer's first sub-batch left in
    // d_part instead of a sum in d_interm (a streamed pass; 0: summed)
    uint32_t last_part_slices = 0;
    // Database-pass timing inside answers (a measurement aid): while
    // time_pass is on, the launches of each sub-batch's database pass (one
    // streamed launch, or its chunks' launches) are bracketed on their
    // stream by events from pass_marks (start, end, start, end, ...).
    static constexpr size_t kMaxPassMarks = 8192;
    bool time_pass = false, time_pass_overflow = false;
    std::vector<hipEvent_t> pass_marks;
    size_t pass_marks_used = 0, passes_timed = 0;
    void mark_pass(hipStream_t s, bool first);
    // Loads of about 1 us: far above any partner skew, bounded so a chain
    // whose partner never runs still ends.
    static constexpr uint32_t kHornerSpinLimit = 1u << 21;
    // Most chains of an answer that run as pairs: a CU for each of their
    // workgroups. 63 steps, all chains in one launch, one workgroup and pair:
    // 541 / 376 us for 1 chain, 555 / 394 for 32, 612 / 464 for 128, 632 / 875
    // for 192 (two workgroups to a CU).
    static constexpr size_t kPairMaxChains = 128;
    // The streamed chains' bound: ~1 s or more of sleeps, far above a
    // database pass's time even queued behind other batches on the device.
    static constexpr uint32_t kStreamSpinLimit = 1u << 23;
    // Enqueue the answer of `count` flat queries at d_in (device) into d_out
    // (device) on stream s, using slots [slot0, slot0 + count) and scratch
    // set `lane` (work that may overlap on the device uses distinct lanes).
    // status_read: the caller reads the lane's status word after the call
    // (check_status): the first kernel clears it.
    void enqueue(const QueryInput& in, size_t count, uint64_t* d_out, hipStream_t s, size_t slot0 = 0,
                 int lane = 0, bool status_read = false);
    // The same wholly on s and the lane's two side streams.
    void enqueue_on(const QueryInput& in, size_t count, uint64_t* d_out, hipStream_t s, size_t slot0, int lane,
                    bool status_read);
    // The pipeline shape of a sub-batch of nq queries where nothing stands
    // against it (capture), and whether an answer has a pipelined sub-batch.
    int shape_for(size_t nq) const;
    bool pipelined(size_t count) const;
    static bool is_capturing(hipStream_t s);
    // Host-staged answer: fill(i, lwe, rest) writes the u32 words of query i's
    // LWE part and of its keys and RGSW rows, each where not null (called from
    // several threads); the flat responses go to out.
    using FillQuery = std::function<void(size_t, uint32_t*, uint32_t*)>;
    void answer_host(size_t count, const FillQuery& fill, uint64_t* out);
    // Whether a staged answer's keys and RGSW rows (43% of a query of 32768
    // rows) go to the device beside the database pass: a serial answer of one
    // sub-batch, with a pass long enough to hide the copy engine's transfer.
    bool late_keys(size_t count) const;
    // enqueue() behind the device wire codecs: count packed queries at d_in
    // (device, qpack_bytes each) -> count*T compressed cts at d_out (device).
    // (stage: a host job still writing them; late: d_in has their LWE parts'
    // bytes alone)
    void enqueue_packed(const uint8_t* d_in, size_t count, uint8_t* d_out, hipStream_t s, size_t slot0 = 0,
                        int lane = 0, bool status_read = false, HostStage* stage = nullptr,
                        const LateKeys* late = nullptr);
    // The LWE parts that ipir_dbg_time_dbpass prepares: those the last call
    // but a flat device one left in the staging (else zeros), wherever it put
    // them.
    QueryInput staged{(const uint64_t*)nullptr};
    size_t staged_stride = 0;
    void set_staged(const QueryInput& in, size_t stride) {
        staged = in;
        staged.stage = nullptr;
        staged.late = nullptr;
        staged_stride = stride;
    }
    // count responses of `bytes` bytes from the pinned staging to out.
    void copy_out(size_t count, size_t bytes, void* out);
    // Host round trip of the packed forms through the pinned staging.
    void answer_packed_host(const uint8_t* in, size_t count, uint8_t* out);
};

// Device bytes of a server: the resident DB and precomp with the fixed
// scratch (twiddles, lanes), what each of max_batch answer slots adds, and
// the peak of gpu_preprocess (DB, precomp and its transient buffers).
// resident_bytes of a server with max_batch B is fixed + B * per_slot.
struct ServerFootprint {
    size_t fixed = 0, per_slot = 0, preprocess_peak = 0;
    size_t part_words = 0;  // row-slice partials per slot (u32 words)
};
ServerFootprint server_footprint(const PublicParams& pp, size_t gchunk);
// Groups per chunk of the pipelined answer by default (about 8 chunks).
size_t default_group_chunk(size_t G);

}  // namespace inspire

// C ABI handle (capi.h): one database generation.
struct ipir_server {
    inspire::PublicParams pp;
    inspire::GpuServerCtx* ctx;
};

// One query's words (a C ABI view), narrowed to u32 as the server stages them.
// The view's words, each part where not null.
void flatten_view(const ipir_query_view& v, size_t R, uint32_t* lwe, uint32_t* rest);
