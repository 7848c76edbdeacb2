// Online (per-query) kernels for gfx950: batched NTT, the row-slice
// reduction of the database pass, pack finalize, and the persistent
// Horner/external-product chain (preparation, database and collapse passes
// live in kernels_prep.hip, kernels_db.hip and kernels_collapse.hip).
//
// Semantics follow the reference's online path (src/gpu_protocol.cu:
// 1121-1339): mat-vec interm_c = DB^T b_c mod q_c (src/gpu_online.cu:23-41);
// per group b = NTT(interm) minus the lazy collapse sums and the final
// D_final x ksk_neg1 term (src/gpu_online.cu:547-632); Horner
// acc = ext_prod(rgsw, acc) + packed[i] (src/gpu_online.cu:474-540). All
// arithmetic is exact, so results equal the reference's bit for bit.
#include "kernels.h"
#include "ntt_regs.h"

namespace ipx {

namespace {

constexpr size_t BLK = (size_t)D_EFF * 2 * N;  // one key / RGSW part, u32 words
// s_sleep argument between two polls of a hand-over counter (units of 64
// clocks); 4, 8, 16 and 32 measured no different from 2 at the 16 GB tier
constexpr int kSpinSleep = 2;

// ------------------------------------------------------------ batched NTT
__global__ __launch_bounds__(256) void k_ntt_rns(uint32_t* __restrict__ polys, NttConst nc, int inverse) {
    __shared__ uint32_t buf[POLY_LDS];
    const int limb = blockIdx.x & 1;
    uint32_t* p = polys + (size_t)blockIdx.x * N;
    const uint32_t t = threadIdx.x;
#pragma unroll
    for (int k = 0; k < 8; k++) buf[ls(t + 256 * k)] = p[t + 256 * k];
    __syncthreads();
    if (inverse) ntt_inv_lds(buf, t, tw_global(nc, limb), limb, nc.inv_n[limb], nc.inv_n_p[limb]);
    else ntt_fwd_lds(buf, t, tw_global(nc, limb), limb);
#pragma unroll
    for (int k = 0; k < 8; k++) p[t + 256 * k] = buf[ls(t + 256 * k)];
}

// ------------------------------------------------------------ slice reduction
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

// interm[q][limb][col] = sum over row slices of part mod q_limb, for columns
// col0 + [0, gridDim.x*256); blockIdx.y = limb, blockIdx.z = query. A
// workgroup covers 256 columns (4 per lane of a wave); its 4 waves take every
// 4th slice, so narrow passes with many slices still spread over many CUs
// and each lane has few loads in sequence. Exact 64-bit sums (< 2^32 per
// slice), combined in LDS, then one reduction.
__global__ __launch_bounds__(256) void k_reduce_slices(const uint32_t* __restrict__ part, size_t part_stride,
                                                       uint32_t S, uint32_t C, uint32_t col0, uint32_t ncols,
                                                       uint32_t* __restrict__ interm) {
    __shared__ uint64_t acc[3][64][4];
    const uint32_t lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const uint32_t j = blockIdx.x * 256 + lane * 4, col = col0 + j;
    const int limb = (int)blockIdx.y;
    const uint32_t q = blockIdx.z;
    const u32x4* pp = reinterpret_cast<const u32x4*>(part + q * part_stride + (size_t)limb * ncols + j);
    const size_t sstride = 2 * (size_t)ncols / 4;  // one slice, in u32x4
    uint64_t a[4] = {0, 0, 0, 0};
#pragma unroll 4
    for (uint32_t s = w; s < S; s += 4) {
        const u32x4 v = __builtin_nontemporal_load(pp + (size_t)s * sstride);
        a[0] += v[0]; a[1] += v[1]; a[2] += v[2]; a[3] += v[3];
    }
    if (w > 0)
#pragma unroll
        for (int e = 0; e < 4; e++) acc[w - 1][lane][e] = a[e];
    __syncthreads();
    if (w > 0) return;
    u32x4 o;
#pragma unroll
    for (int e = 0; e < 4; e++) o[e] = red64(a[e] + acc[0][lane][e] + acc[1][lane][e] + acc[2][lane][e], limb);
    *reinterpret_cast<u32x4*>(interm + (size_t)q * 2 * C + (size_t)limb * C + col) = o;
}

// ------------------------------------------------------------ pack finalize
// packed_b[q][g][c] = NTT(interm[q][c][gN..gN+N-1]) - part2[q][g][c]
//                     - sum_j Df[g][c][j] * Kn[j][c]  (reference
// src/gpu_protocol.cu:1225-1283, src/gpu_online.cu:547-592), where interm is
// the sum of the database pass's row-slice partials (one slice: itself). A
// workgroup per (group, limb, query) of TH lanes: they all sum slices, then
// 256 of them transform in registers (ntt_regs.h). A chain of dependent
// latencies, so every load that depends on nothing (twiddles, Df, Kn, the
// collapse sums) is issued first. Summing here saves a pass over the
// partials and a launch: at 0.13 GB the reduction and the pack took 4.6 +
// 5.6 us and two launches. Where every chain is one ciphertext long (out set)
// the response is written here as well, without a Horner launch (another 5
// us).
template <int TH>
__global__ __launch_bounds__(TH) void k_pack_finalize(const uint32_t* __restrict__ part, size_t part_qstride,
                                                      uint32_t slices, uint32_t C,
                                                      const uint32_t* __restrict__ part2, size_t p2_stride,
                                                      const uint32_t* __restrict__ precomp,
                                                      const uint32_t* __restrict__ keys, size_t kstride,
                                                      uint32_t* __restrict__ packed_b, size_t pstride, uint32_t g0,
                                                      uint64_t* __restrict__ out, NttConst nc) {
    __shared__ __align__(16) uint32_t buf[1][POLY4_LDS];
    const uint32_t g = g0 + blockIdx.x, c = blockIdx.y, qi = blockIdx.z, tid = threadIdx.x, t = tid & 255;
    const bool lead = __builtin_amdgcn_readfirstlane((int)(tid >> 8)) == 0;
    const NrLimb m = nr_limb((int)c);
    const uint32_t* pp = part + (size_t)qi * part_qstride + (size_t)c * C + (size_t)g * N;
    const size_t sstride = 2 * (size_t)C;
    const uint32_t* pc = precomp + (size_t)g * PC_GROUP;
    uint32_t x[1][8];
    NrTw tw[4];
    u32x4 d0[2], d1[2], k0[2], k1[2], s2[2];
    if (lead) {
        nr_tw_global(tw, nc, (int)c, t);
        const u32x4* Df = reinterpret_cast<const u32x4*>(pc + PC_DF + (size_t)c * D_EFF * N + 8 * t);
        const u32x4* Kn =  // key 1 = ksk_neg1, [digit][limb][N]
            reinterpret_cast<const u32x4*>(keys + (size_t)qi * kstride + BLK + (size_t)c * N + 8 * t);
        const u32x4* p2 = reinterpret_cast<const u32x4*>(part2 + (size_t)qi * p2_stride + (size_t)g * 2 * N +
                                                         (size_t)c * N + 8 * t);
#pragma unroll
        for (int h = 0; h < 2; h++) {
            d0[h] = Df[h];
            d1[h] = Df[N / 4 + h];
            k0[h] = Kn[h];
            k1[h] = Kn[2 * N / 4 + h];
            s2[h] = p2[h];
        }
    }
    if (TH == 256) {
        if (slices == 1) {
#pragma unroll
            for (int k = 0; k < 8; k++) x[0][k] = pp[t + 256 * k];
        } else {  // 2..4 slices: up to 32 loads in flight
            uint32_t a[8] = {0, 0, 0, 0, 0, 0, 0, 0};  // residues below 2^27
#pragma unroll
            for (uint32_t s = 0; s < 4; s++)
                if (s < slices)
#pragma unroll
                    for (int k = 0; k < 8; k++) a[k] += pp[s * sstride + t + 256 * k];
#pragma unroll
            for (int k = 0; k < 8; k++) x[0][k] = a[k];  // up to 4q
        }
    } else {
        // lane: 2 columns of every slice, 16 loads in flight
        const u32x2* p = reinterpret_cast<const u32x2*>(pp) + tid;
        uint64_t a0 = 0, a1 = 0;
#pragma unroll 16
        for (uint32_t s = 0; s < slices; s++) {
            const u32x2 v = p[s * (sstride / 2)];
            a0 += v.x;
            a1 += v.y;
        }
        const uint32_t e = 2 * tid, w = e + 4 * (e >> 5);
        *reinterpret_cast<u32x2*>(&buf[0][w]) = u32x2{red64(a0, (int)c), red64(a1, (int)c)};
        __syncthreads();
        if (lead) nr_load<0, 1>(buf, x, t);
    }
    nr_forward1(x, buf, tw, t, m, lead);
    if (lead) {
        u32x4* dst = reinterpret_cast<u32x4*>(packed_b + (size_t)qi * pstride + (size_t)g * 2 * N + (size_t)c * N + 8 * t);
#pragma unroll
        for (int h = 0; h < 2; h++) {
            u32x4 r;
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const uint64_t sub = (uint64_t)d0[h][e] * k0[h][e] + (uint64_t)d1[h][e] * k1[h][e] + s2[h][e];
                const uint32_t v = fold(nr_reduce(x[0][4 * h + e], m), m.q);  // from at most 26q
                r[e] = sub_mod(v, red64(sub, (int)c), m.q);
                x[0][4 * h + e] = r[e];
            }
            dst[h] = r;
        }
    }
    if (!out) return;
    // a chain of one ciphertext: [a|b][limb][N] u64, whole lines through LDS
    if (lead) nr_store<3, 1>(buf, x, t);
    __syncthreads();
    if (!lead) return;
    uint64_t* o = out + (size_t)qi * 4 * N + (size_t)c * N + t;
    const uint32_t* pa = pc + PC_A + (size_t)c * N + t;
#pragma unroll
    for (int k = 0; k < 8; k++) {
        o[256 * k] = pa[256 * k];
        o[2 * N + 256 * k] = buf[0][nr_base(0, t) + nr_stride<0>() * k];
    }
}

// The same result with one workgroup per query: four 256-lane teams take one
// (group, limb) polynomial each per round. A one-query chunk's grid of the
// kernel above (2 workgroups per group) waits for CU slots behind the
// database-pass workgroups running beside it; one workgroup starts as soon
// as one CU has room, like the Horner chain it feeds.
__global__ __launch_bounds__(1024) void k_pack_finalize_wg(const uint32_t* __restrict__ interm, uint32_t C,
                                                           const uint32_t* __restrict__ part2, size_t p2_stride,
                                                           const uint32_t* __restrict__ precomp,
                                                           const uint32_t* __restrict__ keys, size_t kstride,
                                                           uint32_t* __restrict__ packed_b, size_t pstride,
                                                           uint32_t g0, uint32_t ng, NttConst nc) {
    __shared__ uint32_t buf[4][POLY_LDS];
    __shared__ uint32_t twl[8 * N];
    const uint32_t tid = threadIdx.x, team = tid >> 8, t = tid & 255, qi = blockIdx.z;
    const uint32_t npoly = 2 * ng, rounds = (npoly + 3) / 4;
    uint32_t* b = buf[team];
    stage_twiddles(twl, nc, tid, 1024);  // the first round's barrier publishes them
    for (uint32_t r = 0; r < rounds; r++) {  // every lane runs every round (barriers inside)
        const uint32_t k = 4 * r + team;
        const bool active = k < npoly;
        const uint32_t g = g0 + (active ? k >> 1 : 0), c = k & 1;
        const uint32_t q = qof((int)c);
        if (active) {
            const uint32_t* pp = interm + (size_t)qi * 2 * C + (size_t)c * C + (size_t)g * N;
#pragma unroll
            for (int e = 0; e < 8; e++) b[ls(t + 256 * e)] = pp[t + 256 * e];
        }
        __syncthreads();
        ntt_fwd_lds(b, t, tw_lds(twl, (int)c), (int)c, active);
        if (active) {
            const uint32_t* Df = precomp + (size_t)g * PC_GROUP + PC_DF + (size_t)c * D_EFF * N;
            const uint32_t* Kn = keys + qi * kstride + BLK + (size_t)c * N;
            const uint32_t* p2 = part2 + qi * p2_stride + (size_t)g * 2 * N + (size_t)c * N;
#pragma unroll 2
            for (int e = 0; e < 8; e++) {
                const uint32_t i = t + 256 * e;
                const uint64_t sub = (uint64_t)Df[i] * Kn[i] + (uint64_t)Df[N + i] * Kn[2 * N + i] + p2[i];
                packed_b[qi * pstride + (size_t)g * 2 * N + (size_t)c * N + i] =
                    sub_mod(b[ls(i)], red64(sub, (int)c), q);
            }
        }
        __syncthreads();
    }
}

// ------------------------------------------------------------ Horner chain
// One workgroup per (response ciphertext, query), two teams of 256 lanes,
// one per limb. Per step (acc <- ext_prod(rgsw, acc) + packed[i]) a team
// takes its limb's a and b parts from NTT form to coefficients, the teams
// swap halves of the CRT lift through LDS so that each coefficient is
// lifted and cut into digits once, and a team transforms the four digit
// polynomials mod its prime together and multiplies them with the query's
// RGSW rows. A lane holds the same 8 slots of every polynomial at both ends
// of the transforms (ntt_regs.h), so the accumulators, the products and the
// rows stay in registers and a step has 8 barriers. L == 1 copies
// packed[start].
// Bound: VALU issue of one CU (a serial chain; its workgroup has two waves
// per SIMD with the four polynomials as independent work). One team of 256
// lanes per polynomial (16 waves, every transform through LDS with folded
// butterflies, products and digits exchanged through LDS: 20 barriers)
// took 16.6 us per step alone, this form takes 8.7 (two chains of 256 groups
// for 3 queries: 4245 and 2214 us).
// The rows are kept times 2^32 so the four products of a slot are brought
// back with one Montgomery step (2 instructions); the accumulators stay
// below 5q and are made canonical where they leave the kernel.
// The step's packed parts load while the digits are transformed. STREAMED:
// beside a streamed pack the chain needs a group only where it adds the
// group's b-part, so it waits for it (StreamWait) before the step's last
// phase.
struct HornerChain {
    const uint32_t* pa_base;
    size_t pa_stride;
    uint32_t G, Da, T;
    uint32_t* packed_b;
    size_t pstride;
    const uint32_t* rgsw;
    size_t rstride;
    uint64_t* out;
    uint32_t* hstate;
    uint32_t g_lo, g_hi;
    HornerAgain again;
};

template <bool STREAMED>
__global__ __launch_bounds__(512, 2) void k_horner(HornerChain h, NttConst nc, NrGadget gc, FusedPack fp,
                                                   StreamWait sw) {
    __shared__ __align__(16) uint32_t buf[2][4][POLY4_LDS];  // [limb][a, b or the four digit polynomials]
    __shared__ __align__(16) nr_u32x2 tw2[2][N];
    __shared__ uint32_t dx[2][8][2][256];  // digits by the team that made them: [4a + .., 4b + ..][d1, d2][lane]
    __shared__ uint32_t sw_abort;
    const uint32_t ct = blockIdx.x, qi = blockIdx.y, tid = threadIdx.x, t = tid & 255;
    if (!STREAMED && h.again.only_if) {
        if (*h.again.only_if == 0) return;
        if (tid == 0) *h.again.redone = 1;
    }
    const int c = __builtin_amdgcn_readfirstlane((int)(tid >> 8));  // this team's limb
    const uint32_t start = ct * h.Da;
    const uint32_t L = (h.G - start) < h.Da ? (h.G - start) : h.Da;
    const uint32_t top = start + L - 1;
    // this launch covers the chain's groups in [lo, hi), highest first
    const uint32_t lo = start > h.g_lo ? start : h.g_lo, hi = start + L < h.g_hi ? start + L : h.g_hi;
    if (lo >= hi) return;
    const NrLimb m = nr_limb(c);
    // Beside a streamed pack: lane 0 waits until this chain's packed b-part
    // of group g is published (the hand-over rules in dev_common.h); the
    // caller's next barrier publishes sw_abort, set where the wait exceeded
    // its bound.
    const uint32_t* sw_done = sw.done + (size_t)(qi / sw.queries) * sw.stride;
    auto wait_packed = [&](uint32_t g) {
        if (tid == 0) {
            uint32_t spins = 0, ab = 0;
            while (sw.spin_limit == 0 ||
                   __hip_atomic_load(sw_done + g, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == 0) {
                if (++spins > sw.spin_limit) {
                    __hip_atomic_store(sw.status, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    ab = 1;
                    break;
                }
                __builtin_amdgcn_s_sleep(kSpinSleep);
            }
            sw_abort = ab;
        }
    };
    uint64_t* o = h.out + ((size_t)qi * h.T + ct) * 4 * N;
    auto poison = [&]() {  // an invalid response: no residue is all-ones
        for (uint32_t x = tid; x < 4 * N; x += 512) o[x] = ~0ull;
    };
    uint32_t* pbw = h.packed_b + qi * h.pstride;
    if (fp.interm) {
        // this chain's packed b-parts of groups [lo, hi), team c the limb c
        // (as k_pack_finalize): written to packed_b and read back below
        // after the block's barrier
        const Tw gtw = tw_global(nc, c);
        uint32_t* b = buf[c][0];
        for (uint32_t g = lo; g < hi; g++) {  // every lane runs every round (barriers inside)
            const uint32_t* src = fp.interm + (size_t)qi * 2 * fp.C + (size_t)c * fp.C + (size_t)g * N;
#pragma unroll
            for (int e = 0; e < 8; e++) b[ls(t + 256 * e)] = src[t + 256 * e];
            __syncthreads();
            ntt_fwd_lds(b, t, gtw, c);
            const uint32_t* Df = fp.precomp + (size_t)g * PC_GROUP + PC_DF + (size_t)c * D_EFF * N;
            const uint32_t* Kn = fp.keys + qi * fp.keys_stride + BLK + (size_t)c * N;
            const uint32_t* p2 = fp.part2 + qi * fp.part2_stride + (size_t)g * 2 * N + (size_t)c * N;
#pragma unroll 2
            for (int e = 0; e < 8; e++) {
                const uint32_t i = t + 256 * e;
                const uint64_t sub = (uint64_t)Df[i] * Kn[i] + (uint64_t)Df[N + i] * Kn[2 * N + i] + p2[i];
                pbw[(size_t)g * 2 * N + (size_t)c * N + i] = sub_mod(b[ls(i)], red64(sub, c), m.q);
            }
            __syncthreads();
        }
    }
    const uint32_t* pb = pbw;
    const uint32_t* rg = h.rgsw + qi * h.rstride;
    uint32_t* hs = h.hstate + ((size_t)qi * h.T + ct) * 4 * N;  // chain state between launches
    // 8 consecutive slots of this lane's limb
    auto load8 = [&](uint32_t (&x)[8], const uint32_t* p) {
        const u32x4* s = reinterpret_cast<const u32x4*>(p + (size_t)c * N + 8 * t);
        const u32x4 l = s[0], u = s[1];
#pragma unroll
        for (int k = 0; k < 4; k++) {
            x[k] = l[k];
            x[k + 4] = u[k];
        }
    };
    // the same of a b-part: handed over by a streamed pack, or ordinary
    auto load8b = [&](uint32_t (&x)[8], const uint32_t* p) {
        if constexpr (STREAMED) {
#pragma unroll
            for (int k = 0; k < 4; k++) {
                const uint64_t v = agent_load2(p + (size_t)c * N + 8 * t + 2 * k);
                x[2 * k] = (uint32_t)v;
                x[2 * k + 1] = (uint32_t)(v >> 32);
            }
        } else {
            load8(x, p);
        }
    };
    uint32_t acc[2][8];  // a and b part, slots 8t + k
    int first;
    if (top < h.g_hi) {  // the chain starts here: acc = packed[top]
        if constexpr (STREAMED) {
            wait_packed(top);
            __syncthreads();
            if (sw_abort) {
                poison();
                return;
            }
        }
        load8(acc[0], h.pa_base + (size_t)top * h.pa_stride);
        load8b(acc[1], pb + (size_t)top * 2 * N);
        first = (int)top - 1;
    } else {
        load8(acc[0], hs);
        load8(acc[1], hs + 2 * N);
        first = (int)hi - 1;
    }
    if (first >= (int)lo) {
        nr_stage_twiddles(tw2, nc, tid, 512);  // published by the barrier below
        // the query's rows of this limb, [top_a | top_b | bot_a | bot_b][digit][slot], times 2^32 mod q
        const uint32_t r32 = c ? (uint32_t)(4294967296ull % Q1) : (uint32_t)(4294967296ull % Q0);
        const uint32_t qneg = c ? nr_neg_inverse(Q1) : nr_neg_inverse(Q0);
        uint32_t rows[4][2][8];
#pragma unroll
        for (int p = 0; p < 4; p++)
#pragma unroll
            for (int j = 0; j < 2; j++) {
                load8(rows[p][j], rg + (size_t)p * BLK + (size_t)j * 2 * N);
#pragma unroll
                for (int k = 0; k < 8; k++) rows[p][j][k] = mul_mod(rows[p][j][k], r32, c);
            }
        const nr_u32x2* tw = tw2[c];
        uint32_t(*xs)[256] = reinterpret_cast<uint32_t(*)[256]>(buf[c][2]);            // lift shares sent
        const uint32_t(*xr)[256] = reinterpret_cast<const uint32_t(*)[256]>(buf[1 - c][2]);  // and received
        __syncthreads();
        for (int gs = first; gs >= (int)lo; gs--) {
            uint32_t cf[2][8];  // a and b part, coefficients t + 256k
#pragma unroll
            for (int p = 0; p < 2; p++)
#pragma unroll
                for (int k = 0; k < 8; k++) cf[p][k] = acc[p][k];
            nr_inverse<2>(cf, buf[c], tw, t, m);
            // this limb's shares of the CRT lift; team c lifts the
            // coefficients k in [4c, 4c + 4) and sends the others
            uint32_t keep[2][4];
#pragma unroll
            for (int p = 0; p < 2; p++)
#pragma unroll
                for (int k = 0; k < 8; k++) cf[p][k] = nr_crt_part(cf[p][k], gc, c, m);
#pragma unroll
            for (int p = 0; p < 2; p++)
#pragma unroll
                for (int k = 0; k < 4; k++) {
                    keep[p][k] = c ? cf[p][k + 4] : cf[p][k];
                    xs[4 * p + k][t] = c ? cf[p][k] : cf[p][k + 4];
                }
            lds_barrier();
            uint32_t x[4][8];  // digit polynomials a1, a2, b1, b2: residues + q mod this limb's prime
#pragma unroll
            for (int p = 0; p < 2; p++)
#pragma unroll
                for (int k = 0; k < 4; k++) {
                    const uint32_t other = xr[4 * p + k][t];
                    const nr_u32x2 d = nr_digits(c ? other : keep[p][k], c ? keep[p][k] : other);
                    dx[c][4 * p + k][0][t] = d.x;
                    dx[c][4 * p + k][1][t] = d.y;
                }
            lds_barrier();
            uint32_t pav[8], pbv[8];  // the step's packed parts, in flight during the transforms
            load8(pav, h.pa_base + (size_t)gs * h.pa_stride);
            if constexpr (!STREAMED) load8(pbv, pb + (size_t)gs * 2 * N);
#pragma unroll
            for (int p = 0; p < 2; p++)
#pragma unroll
                for (int s = 0; s < 2; s++)
#pragma unroll
                    for (int k = 0; k < 4; k++) {
                        x[2 * p][4 * s + k] = dx[s][4 * p + k][0][t] + (m.q - (1u << 17));
                        x[2 * p + 1][4 * s + k] = dx[s][4 * p + k][1][t] + m.q;
                    }
            nr_forward<4>(x, buf[c], tw, t, m, [&]() {
                if constexpr (STREAMED) {
                    wait_packed((uint32_t)gs);
                    __syncthreads();  // no wave's load of the b-part before the flag was seen
                } else {
                    lds_barrier();
                }
            });
            if constexpr (STREAMED) {
                if (sw_abort) {
                    poison();
                    return;
                }
                load8b(pbv, pb + (size_t)gs * 2 * N);
            }
#pragma unroll
            for (int k = 0; k < 8; k++) {
                // digits below 23.1q, rows below q: the sums stay below 93 q^2 < 2^59.6
                uint64_t sa = 0, sb = 0;
#pragma unroll
                for (int s = 0; s < 2; s++)
#pragma unroll
                    for (int j = 0; j < 2; j++) {
                        sa += (uint64_t)x[2 * s + j][k] * rows[2 * s][j][k];
                        sb += (uint64_t)x[2 * s + j][k] * rows[2 * s + 1][j][k];
                    }
                acc[0][k] = nr_montgomery(sa, qneg, m.q) + pav[k];  // below 2.1q + q + q
                acc[1][k] = nr_montgomery(sb, qneg, m.q) + pbv[k];
            }
        }
#pragma unroll
        for (int p = 0; p < 2; p++)
#pragma unroll
            for (int k = 0; k < 8; k++) acc[p][k] = fold(fold(fold(acc[p][k], 4 * m.q), 2 * m.q), m.q);
    }
    if (lo > start) {  // the chain continues in a later launch
#pragma unroll
        for (int p = 0; p < 2; p++) {
            u32x4* d = reinterpret_cast<u32x4*>(hs + (size_t)(2 * p + c) * N + 8 * t);
            d[0] = u32x4{acc[p][0], acc[p][1], acc[p][2], acc[p][3]};
            d[1] = u32x4{acc[p][4], acc[p][5], acc[p][6], acc[p][7]};
        }
        return;
    }
    // the response, through LDS for whole lines of 8-byte words (a lane's own
    // words of the last exchange)
    nr_store<3, 2>(buf[c], acc, t);
    __syncthreads();
#pragma unroll
    for (int p = 0; p < 2; p++)
#pragma unroll
        for (int k = 0; k < 8; k++)
            o[(size_t)(2 * p + c) * N + t + 256 * k] = buf[c][p][nr_base(0, t) + nr_stride<0>() * k];
}

// ------------------------------------------------------------ streamed pack
// Beside a streamed database pass (launch_pack_stream): workgroup b packs
// queries [b*ps.queries, ...) group by group from the top; team k of
// round r takes polynomial 4r + k = (query, limb), the limb of its own
// twiddles, and transforms it in registers (ntt_regs.h). Df x Kn of round 0
// (in place before the launch) is computed while lane 0 waits for the group;
// the partials and the collapse sums are read at agent scope, all of a
// lane's in flight together.
__global__ __launch_bounds__(1024) void k_pack_stream(PackStream ps, const uint32_t* __restrict__ part2,
                                                      size_t p2_stride, const uint32_t* __restrict__ precomp,
                                                      const uint32_t* __restrict__ keys, size_t kstride,
                                                      uint32_t* __restrict__ packed_b, size_t pstride, uint32_t G,
                                                      uint32_t nq, NttConst nc) {
    __shared__ __align__(16) uint32_t buf[4][1][POLY4_LDS];
    __shared__ __align__(16) nr_u32x2 tw2[2][N];
    __shared__ uint32_t abort_flag;
    const uint32_t tid = threadIdx.x, t = tid & 255, blk = blockIdx.x;
    if (ps.only_if && *ps.only_if == 0) return;
    const uint32_t team = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid >> 8));
    const uint32_t q0 = blk * ps.queries;
    const uint32_t nqb = nq - q0 < ps.queries ? nq - q0 : ps.queries;
    const uint32_t npoly = 2 * nqb, rounds = (npoly + 3) / 4;
    const int c = (int)(team & 1);
    const NrLimb m = nr_limb(c);
    const size_t sstride = 2 * (size_t)ps.C;  // one row slice of the pass's partials
    nr_stage_twiddles(tw2, nc, tid, 1024);    // published by the first barrier below
    for (int g = (int)G - 1; g >= 0; g--) {
        for (uint32_t r = 0; r < rounds; r++) {  // every lane runs every round (barriers inside)
            const uint32_t k = 4 * r + team;
            const bool active = k < npoly;
            const uint32_t qi = q0 + (active ? k >> 1 : 0);
            uint32_t sub[8];
            if (active) {
                const u32x4* Df = reinterpret_cast<const u32x4*>(precomp + (size_t)g * PC_GROUP + PC_DF +
                                                                 (size_t)c * D_EFF * N + 8 * t);
                const u32x4* Kn =
                    reinterpret_cast<const u32x4*>(keys + (size_t)qi * kstride + BLK + (size_t)c * N + 8 * t);
#pragma unroll
                for (int h = 0; h < 2; h++) {
                    const u32x4 d0 = Df[h], d1 = Df[N / 4 + h], k0 = Kn[h], k1 = Kn[2 * N / 4 + h];
#pragma unroll
                    for (int e = 0; e < 4; e++)
                        sub[4 * h + e] = red64((uint64_t)d0[e] * k0[e] + (uint64_t)d1[e] * k1[e], c);
                }
            }
            if (r == 0) {
                if (tid == 0) {
                    uint32_t spins = 0, ab = 0;
                    while (ps.spin_limit == 0 || __hip_atomic_load(ps.pass_done + g, __ATOMIC_RELAXED,
                                                                   __HIP_MEMORY_SCOPE_AGENT) < ps.pass_target) {
                        if (++spins > ps.spin_limit) {
                            __hip_atomic_store(ps.status, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                            ab = 1;
                            break;
                        }
                        __builtin_amdgcn_s_sleep(kSpinSleep);
                    }
                    abort_flag = ab;
                }
                __syncthreads();  // no wave's load of the partials before the count was seen
                if (abort_flag) return;
            }
            uint32_t x[1][8];
            if (active) {
                // columns 2t + 512k (a pair each) of every slice: residues below
                // 2^27, at most 16 of them, so 32-bit sums below 16q
                const uint32_t* src = ps.part + qi * ps.part_qstride + (size_t)c * ps.C + (size_t)g * N + 2 * t;
                const uint32_t* p2 = part2 + qi * p2_stride + (size_t)g * 2 * N + (size_t)c * N + 8 * t;
                uint32_t a[8] = {0, 0, 0, 0, 0, 0, 0, 0};
                uint64_t s2[4];
#pragma unroll
                for (int e = 0; e < 4; e++) s2[e] = agent_load2(p2 + 2 * e);
#pragma unroll 4
                for (uint32_t sl = 0; sl < ps.slices; sl++)
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        const uint64_t v = agent_load2(src + sl * sstride + 512 * e);
                        a[2 * e] += (uint32_t)v;
                        a[2 * e + 1] += (uint32_t)(v >> 32);
                    }
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    const uint32_t col = 2 * t + 512 * e;
                    *reinterpret_cast<u32x2*>(&buf[team][0][col + 4 * (col >> 5)]) = u32x2{a[2 * e], a[2 * e + 1]};
                    sub[2 * e] = red64((uint64_t)sub[2 * e] + (uint32_t)s2[e], c);
                    sub[2 * e + 1] = red64((uint64_t)sub[2 * e + 1] + (uint32_t)(s2[e] >> 32), c);
                }
            }
            lds_barrier();
            if (active) nr_load<0, 1>(buf[team], x, t);
            nr_forward<1>(x, buf[team], tw2[c], t, m, [] { lds_barrier(); });  // from 16q: below 38q
            if (active) {
                uint32_t* dst = packed_b + qi * pstride + (size_t)g * 2 * N + (size_t)c * N + 8 * t;
#pragma unroll
                for (int e = 0; e < 8; e++) x[0][e] = sub_mod(fold(nr_reduce(x[0][e], m), m.q), sub[e], m.q);
#pragma unroll
                for (int e = 0; e < 4; e++) agent_store2(dst + 2 * e, x[0][2 * e], x[0][2 * e + 1]);
            }
            lds_barrier();  // the buffers are free for the next round
        }
        // publish the group once every wave's stores are complete
        __builtin_amdgcn_s_waitcnt(0);
        __syncthreads();
        if (tid == 0)
            __hip_atomic_store(ps.packed_done + (size_t)blk * G + g, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
}

}  // namespace

namespace {
// Plain grid-stride copy, 16 bytes per lane: the reference point that
// scales the memory-traffic counters of the other kernels.
__global__ __launch_bounds__(256) void k_copy16(const u32x4* __restrict__ src, u32x4* __restrict__ dst, size_t n) {
    for (size_t x = (size_t)blockIdx.x * 256 + threadIdx.x; x < n; x += (size_t)gridDim.x * 256)
        dst[x] = __builtin_nontemporal_load(src + x);
}
}  // namespace

hipError_t launch_copy16(const void* src, void* dst, size_t bytes, hipStream_t s) {
    if (bytes % 16) return hipErrorInvalidValue;
    if (bytes == 0) return hipSuccess;
    hipLaunchKernelGGL(k_copy16, dim3(8192), dim3(256), 0, s, static_cast<const u32x4*>(src), static_cast<u32x4*>(dst),
                       bytes / 16);
    return hipGetLastError();
}

hipError_t launch_ntt_rns(uint32_t* polys, size_t npoly, const NttConst& nc, bool inverse, hipStream_t s) {
    if (npoly == 0) return hipSuccess;
    hipLaunchKernelGGL(k_ntt_rns, dim3((unsigned)(2 * npoly)), dim3(256), 0, s, polys, nc, inverse ? 1 : 0);
    return hipGetLastError();
}

hipError_t launch_reduce_slices(const uint32_t* part, size_t part_stride, uint32_t S, size_t C, uint32_t* interm,
                                size_t nq, size_t col0, size_t ncols, hipStream_t s) {
    if (ncols % 1024 || col0 % 4 || col0 + ncols > C) return hipErrorInvalidValue;
    if (nq == 0 || ncols == 0) return hipSuccess;
    hipLaunchKernelGGL(k_reduce_slices, dim3((unsigned)(ncols / 256), 2, (unsigned)nq), dim3(256), 0, s, part,
                       part_stride, S, (uint32_t)C, (uint32_t)col0, (uint32_t)ncols, interm);
    return hipGetLastError();
}

hipError_t launch_pack_finalize(const uint32_t* part, size_t part_qstride, uint32_t slices, size_t C,
                                const uint32_t* part2, size_t part2_stride, const uint32_t* precomp, size_t g0,
                                size_t ng, const uint32_t* keys, size_t keys_stride, uint32_t* packed_b,
                                size_t packed_stride, size_t nq, const NttConst& nc, hipStream_t s, uint64_t* out) {
    if (ng == 0 || nq == 0) return hipSuccess;
    if (slices == 0 || (out && (g0 != 0 || ng != 1 || C != N))) return hipErrorInvalidValue;
    const dim3 grid((unsigned)ng, 2, (unsigned)nq);
    // from 5 slices on the sums take 1024 lanes
    if (slices > 4)
        hipLaunchKernelGGL(k_pack_finalize<1024>, grid, dim3(1024), 0, s, part, part_qstride, slices, (uint32_t)C, part2,
                           part2_stride, precomp, keys, keys_stride, packed_b, packed_stride, (uint32_t)g0, out, nc);
    else
        hipLaunchKernelGGL(k_pack_finalize<256>, grid, dim3(256), 0, s, part, part_qstride, slices, (uint32_t)C, part2,
                           part2_stride, precomp, keys, keys_stride, packed_b, packed_stride, (uint32_t)g0, out, nc);
    return hipGetLastError();
}

hipError_t launch_pack_finalize_wg(const uint32_t* interm, size_t C, const uint32_t* part2, size_t part2_stride,
                                   const uint32_t* precomp, size_t g0, size_t ng, const uint32_t* keys,
                                   size_t keys_stride, uint32_t* packed_b, size_t packed_stride, size_t nq,
                                   const NttConst& nc, hipStream_t s) {
    if (ng == 0 || nq == 0) return hipSuccess;
    hipLaunchKernelGGL(k_pack_finalize_wg, dim3(1, 1, (unsigned)nq), dim3(1024), 0, s, interm, (uint32_t)C, part2,
                       part2_stride, precomp, keys, keys_stride, packed_b, packed_stride, (uint32_t)g0, (uint32_t)ng,
                       nc);
    return hipGetLastError();
}

hipError_t launch_pack_stream(const PackStream& ps, const uint32_t* part2, size_t part2_stride,
                              const uint32_t* precomp, const uint32_t* keys, size_t keys_stride, uint32_t* packed_b,
                              size_t packed_stride, size_t G, size_t nq, const NttConst& nc, hipStream_t s) {
    if (nq == 0 || G == 0) return hipSuccess;
    if (!ps.part || !ps.pass_done || !ps.packed_done || !ps.status || ps.slices == 0 || ps.slices > 16 ||
        ps.C < G * N || ps.queries == 0 || ps.queries > kPackQueries)  // at most 16 partials below 2^27 keep
        return hipErrorInvalidValue;                                    // the 32-bit sums exact
    const unsigned blocks = (unsigned)((nq + ps.queries - 1) / ps.queries);
    hipLaunchKernelGGL(k_pack_stream, dim3(blocks), dim3(1024), 0, s, ps, part2, part2_stride, precomp, keys,
                       keys_stride, packed_b, packed_stride, (uint32_t)G, (uint32_t)nq, nc);
    return hipGetLastError();
}

hipError_t launch_horner(const uint32_t* pa_base, size_t pa_stride, size_t G, size_t Da, size_t T,
                         uint32_t* packed_b, size_t packed_stride, const uint32_t* rgsw, size_t rgsw_stride,
                         uint64_t* out, uint32_t* hstate, size_t g_lo, size_t g_hi, size_t nq, const NttConst& nc,
                         const CrtConst& cc, hipStream_t s, const FusedPack& pack, const StreamWait& wait,
                         const HornerAgain& again) {
    if (nq == 0 || g_lo >= g_hi) return hipSuccess;
    if (wait.done && (!wait.status || wait.queries == 0)) return hipErrorInvalidValue;
    if (again.only_if && (!again.redone || wait.done || pack.interm)) return hipErrorInvalidValue;
    const HornerChain h{pa_base, pa_stride, (uint32_t)G, (uint32_t)Da, (uint32_t)T, packed_b, packed_stride,
                        rgsw, rgsw_stride, out, hstate, (uint32_t)g_lo, (uint32_t)g_hi, again};
    const NrGadget gc = nr_gadget_const(nc, cc);
    const dim3 grid((unsigned)T, (unsigned)nq);
    if (wait.done)
        hipLaunchKernelGGL(k_horner<true>, grid, dim3(512), 0, s, h, nc, gc, pack, wait);
    else
        hipLaunchKernelGGL(k_horner<false>, grid, dim3(512), 0, s, h, nc, gc, pack, wait);
    return hipGetLastError();
}

}  // namespace ipx
