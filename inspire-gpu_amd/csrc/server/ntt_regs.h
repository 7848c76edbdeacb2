// Negacyclic transforms kept in registers between their exchanges: a team
// of 256 lanes transforms P polynomials of one limb at once, each lane
// holding 8 coefficients of every polynomial, with three exchanges through
// LDS (radix-8, -8, -8, -4). Used where a kernel runs transforms back to
// back, so a transform's inputs and outputs never go through LDS and its
// twiddles are read once for all P polynomials.
//
// What bounds it is the VALU: on gfx950 32-bit multiplies, v_mad_u64_u32
// and adds issue at the same rate (4.6-5.5 cycles per wave instruction and
// SIMD, launch included), so instructions are what counts. A butterfly is
// 5 of them here (mul_hi, two v_mad_u64_u32 whose low words are
// u + x*w - t*q, one shift-add, one subtract): 26.7 cycles per wave
// butterfly against 40.9 for the folded form (9 instructions) and 31.9
// without its fold. No fold is needed: q < 2^26.51 leaves 45 q below 2^32,
// and a forward transform grows its inputs by 2q per stage, 22q in all. The
// inverse doubles sums, so the few values that could pass 4q are brought
// back between its phases (2 instructions each).
#pragma once
#include "dev_common.h"

namespace ipx {

typedef uint32_t nr_u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t nr_u32x4 __attribute__((ext_vector_type(4)));

// LDS slot of coefficient e: four pad words per 32 keep 16-byte alignment
// for the radix-4 phase (8 consecutive coefficients per lane) and put the
// stride-4 phase's 8 groups of 4 lanes on 32 different banks.
constexpr uint32_t POLY4_LDS = N + N / 8;

// a*b + c (low words; the high halves of c and of the result are unused)
__device__ __forceinline__ nr_u32x2 nr_mad(uint32_t a, uint32_t b, nr_u32x2 c) {
    nr_u32x2 d;
    uint64_t carry;
    asm("v_mad_u64_u32 %0, %1, %2, %3, %4" : "=v"(d), "=s"(carry) : "v"(a), "v"(b), "v"(c));
    return d;
}
__device__ __forceinline__ nr_u32x2 nr_mad_s(uint32_t a, uint32_t b_uniform, nr_u32x2 c) {
    nr_u32x2 d;
    uint64_t carry;
    asm("v_mad_u64_u32 %0, %1, %2, %3, %4" : "=v"(d), "=s"(carry) : "v"(a), "s"(b_uniform), "v"(c));
    return d;
}
__device__ __forceinline__ nr_u32x2 nr_low(uint32_t x) {
    nr_u32x2 p;
    p.x = x;
    return p;  // p.y: never read
}

// Constants of one limb (uniform over the wave).
struct NrLimb {
    uint32_t q, nq;  // q and 2^32 - q
};
__device__ __forceinline__ NrLimb nr_limb(int c) { return NrLimb{qof(c), 0u - qof(c)}; }

// x*w mod q up to one extra q (below 2q), any x < 2^32.
__device__ __forceinline__ uint32_t nr_mul(uint32_t x, uint32_t w, uint32_t wp, const NrLimb& m) {
    return nr_mad_s(mulhi32(x, wp), m.nq, nr_low(x * w)).x;
}
// x mod q up to a little more than q (below 1.5q) for any x < 2^32:
// floor(2^32/q) = 45 for both primes.
__device__ __forceinline__ uint32_t nr_reduce(uint32_t x, const NrLimb& m) {
    return nr_mad_s(mulhi32(x, 45u), m.nq, nr_low(x)).x;
}
static_assert(4294967296ull / Q0 == 45 && 4294967296ull / Q1 == 45, "45q is the headroom of the lazy transforms");

// Forward butterfly: (u, y) -> (u + y*w, u - y*w + 2q), both 2q above u's bound.
__device__ __forceinline__ void nr_fwd_bf(uint32_t& u, uint32_t& y, nr_u32x2 w, const NrLimb& m) {
    const nr_u32x2 s = nr_mad_s(mulhi32(y, w.y), m.nq, nr_mad(y, w.x, nr_low(u)));
    y = (u << 1) + 2 * m.q - s.x;
    u = s.x;
}
// Inverse butterfly with u <= B q: (u, v) -> (u + v, (v - u)*w mod q below 2q).
// The inverse twiddle psi^-e equals -psi^(N-e), a forward table entry
// negated (nr_inv_index), which swaps the difference.
template <uint32_t B>
__device__ __forceinline__ void nr_inv_bf(uint32_t& u, uint32_t& v, nr_u32x2 w, const NrLimb& m) {
    const uint32_t d = v + (B * m.q - u);
    u = u + v;
    v = nr_mul(d, w.x, w.y, m);
}

// Twiddles of the 8 coefficients of table node A (stages of 1, 2 and 4
// nodes): the forward table of the limb as (w, companion) pairs in LDS.
struct NrTw {
    nr_u32x2 a, b[2], c[4];
};
__device__ __forceinline__ void nr_tw_load(NrTw& t, const nr_u32x2* tw, uint32_t A, bool top) {
    if (top) t.a = tw[A];
    const nr_u32x4* t4 = reinterpret_cast<const nr_u32x4*>(tw);
    const nr_u32x4 b = t4[A], c0 = t4[2 * A], c1 = t4[2 * A + 1];
    t.b[0] = b.xy;
    t.b[1] = b.zw;
    t.c[0] = c0.xy;
    t.c[1] = c0.zw;
    t.c[2] = c1.xy;
    t.c[3] = c1.zw;
}

// One forward phase on a lane's 8 coefficients per polynomial (TOP: three
// stages, else the two lower ones).
template <int P, bool TOP>
__device__ __forceinline__ void nr_fwd_phase(uint32_t (&x)[P][8], const NrTw& t, const NrLimb& m) {
    if (TOP)
#pragma unroll
        for (int k = 0; k < 4; k++)
#pragma unroll
            for (int p = 0; p < P; p++) nr_fwd_bf(x[p][k], x[p][k + 4], t.a, m);
#pragma unroll
    for (int h = 0; h < 2; h++)
#pragma unroll
        for (int k = 4 * h; k < 4 * h + 2; k++)
#pragma unroll
            for (int p = 0; p < P; p++) nr_fwd_bf(x[p][k], x[p][k + 2], t.b[h], m);
#pragma unroll
    for (int h = 0; h < 4; h++)
#pragma unroll
        for (int p = 0; p < P; p++) nr_fwd_bf(x[p][2 * h], x[p][2 * h + 1], t.c[h], m);
}

// One inverse phase with inputs up to B0 q (t: the mirrored node's twiddles).
template <int P, bool TOP, uint32_t B0>
__device__ __forceinline__ void nr_inv_phase(uint32_t (&x)[P][8], const NrTw& t, const NrLimb& m) {
    static_assert((TOP ? 8 : 4) * B0 <= 32, "sums stay below 2^32");
#pragma unroll
    for (int h = 0; h < 4; h++)
#pragma unroll
        for (int p = 0; p < P; p++) nr_inv_bf<B0>(x[p][2 * h], x[p][2 * h + 1], t.c[3 - h], m);
#pragma unroll
    for (int h = 0; h < 2; h++)
#pragma unroll
        for (int k = 4 * h; k < 4 * h + 2; k++)
#pragma unroll
            for (int p = 0; p < P; p++) nr_inv_bf<2 * B0>(x[p][k], x[p][k + 2], t.b[1 - h], m);
    if (TOP)
#pragma unroll
        for (int k = 0; k < 4; k++)
#pragma unroll
            for (int p = 0; p < P; p++) nr_inv_bf<4 * B0>(x[p][k], x[p][k + 4], t.a, m);
}

// Table node of lane t in each phase: coefficients t + 256k, then strides
// 32, 4 and 1 (8t + k).
__device__ __forceinline__ uint32_t nr_node(int phase, uint32_t t) {
    return phase == 0 ? 1u : phase == 1 ? 8 + (t >> 5) : phase == 2 ? 64 + (t >> 2) : 256 + t;
}
// The node whose negated twiddles are the inverse ones: entry m + g of the
// inverse table is minus entry 2m - 1 - g of the forward table.
__device__ __forceinline__ uint32_t nr_inv_node(int phase, uint32_t t) {
    return phase == 0 ? 1u : phase == 1 ? 15 - (t >> 5) : phase == 2 ? 127 - (t >> 2) : 511 - t;
}

// First LDS word of lane t's 8 coefficients in each phase, and their stride.
__device__ __forceinline__ uint32_t nr_base(int phase, uint32_t t) {
    return phase == 0   ? t + 4 * (t >> 5)
           : phase == 1 ? 288 * (t >> 5) + (t & 31)
           : phase == 2 ? 36 * (t >> 2) + (t & 3)
                        : 8 * t + 4 * (t >> 2);
}
template <int PHASE>
constexpr uint32_t nr_stride() {
    return PHASE == 0 ? 288 : PHASE == 1 ? 36 : PHASE == 2 ? 4 : 1;
}

template <int PHASE, int P>
__device__ __forceinline__ void nr_store(uint32_t (*buf)[POLY4_LDS], const uint32_t (&x)[P][8], uint32_t t) {
    const uint32_t b = nr_base(PHASE, t);
#pragma unroll
    for (int p = 0; p < P; p++) {
        if (PHASE == 3) {
            nr_u32x4* d = reinterpret_cast<nr_u32x4*>(&buf[p][b]);
            d[0] = nr_u32x4{x[p][0], x[p][1], x[p][2], x[p][3]};
            d[1] = nr_u32x4{x[p][4], x[p][5], x[p][6], x[p][7]};
        } else {
#pragma unroll
            for (int k = 0; k < 8; k++) buf[p][b + nr_stride<PHASE>() * k] = x[p][k];
        }
    }
}
template <int PHASE, int P>
__device__ __forceinline__ void nr_load(uint32_t (*buf)[POLY4_LDS], uint32_t (&x)[P][8], uint32_t t) {
    const uint32_t b = nr_base(PHASE, t);
#pragma unroll
    for (int p = 0; p < P; p++) {
        if (PHASE == 3) {
            const nr_u32x4* s = reinterpret_cast<const nr_u32x4*>(&buf[p][b]);
            const nr_u32x4 l = s[0], h = s[1];
#pragma unroll
            for (int k = 0; k < 4; k++) {
                x[p][k] = l[k];
                x[p][k + 4] = h[k];
            }
        } else {
#pragma unroll
            for (int k = 0; k < 8; k++) x[p][k] = buf[p][b + nr_stride<PHASE>() * k];
        }
    }
}

// Forward transform of P polynomials: in, coefficients t + 256k (up to
// B q, B <= 23); out, NTT slots 8t + k up to (B + 22) q. buf: the team's P
// LDS polynomials, whose words t + 256k (all lanes' own) must be free; the
// workgroup runs it together (three barriers, the third one last_barrier()).
template <int P, typename F>
__device__ __forceinline__ void nr_forward(uint32_t (&x)[P][8], uint32_t (*buf)[POLY4_LDS], const nr_u32x2* tw,
                                           uint32_t t, const NrLimb& m, F&& last_barrier) {
    NrTw w;
    nr_tw_load(w, tw, nr_node(0, t), true);
    nr_fwd_phase<P, true>(x, w, m);
    nr_store<0, P>(buf, x, t);
    nr_tw_load(w, tw, nr_node(1, t), true);
    lds_barrier();
    nr_load<1, P>(buf, x, t);
    nr_fwd_phase<P, true>(x, w, m);
    nr_store<1, P>(buf, x, t);
    nr_tw_load(w, tw, nr_node(2, t), true);
    lds_barrier();
    nr_load<2, P>(buf, x, t);
    nr_fwd_phase<P, true>(x, w, m);
    nr_store<2, P>(buf, x, t);
    nr_tw_load(w, tw, nr_node(3, t), false);
    last_barrier();
    nr_load<3, P>(buf, x, t);
    nr_fwd_phase<P, false>(x, w, m);
}

// The four phases' twiddles of lane t from the device tables, all loads in
// flight together: for kernels that transform one polynomial and leave.
__device__ __forceinline__ void nr_tw_global(NrTw (&w)[4], const NttConst& nc, int c, uint32_t t) {
    const uint32_t* f = nc.tw + (size_t)c * 4 * N;
    const uint32_t* fp = f + N;
#pragma unroll
    for (int ph = 0; ph < 4; ph++) {
        const uint32_t A = nr_node(ph, t);
        const nr_u32x2 b = *reinterpret_cast<const nr_u32x2*>(f + 2 * A);
        const nr_u32x2 bp = *reinterpret_cast<const nr_u32x2*>(fp + 2 * A);
        const nr_u32x4 q = *reinterpret_cast<const nr_u32x4*>(f + 4 * A);
        const nr_u32x4 qp = *reinterpret_cast<const nr_u32x4*>(fp + 4 * A);
        if (ph < 3) w[ph].a = nr_u32x2{f[A], fp[A]};
#pragma unroll
        for (int h = 0; h < 2; h++) w[ph].b[h] = nr_u32x2{b[h], bp[h]};
#pragma unroll
        for (int h = 0; h < 4; h++) w[ph].c[h] = nr_u32x2{q[h], qp[h]};
    }
}
// Forward transform of one polynomial with those twiddles (bounds and
// layout as nr_forward; every lane of the workgroup calls it, lanes of other
// teams with active = false).
__device__ __forceinline__ void nr_forward1(uint32_t (&x)[1][8], uint32_t (*buf)[POLY4_LDS], const NrTw (&w)[4],
                                            uint32_t t, const NrLimb& m, bool active = true) {
    if (active) {
        nr_fwd_phase<1, true>(x, w[0], m);
        nr_store<0, 1>(buf, x, t);
    }
    lds_barrier();
    if (active) {
        nr_load<1, 1>(buf, x, t);
        nr_fwd_phase<1, true>(x, w[1], m);
        nr_store<1, 1>(buf, x, t);
    }
    lds_barrier();
    if (active) {
        nr_load<2, 1>(buf, x, t);
        nr_fwd_phase<1, true>(x, w[2], m);
        nr_store<2, 1>(buf, x, t);
    }
    lds_barrier();
    if (active) {
        nr_load<3, 1>(buf, x, t);
        nr_fwd_phase<1, false>(x, w[3], m);
    }
}

// Inverse transform without its N^-1 scale: in, NTT slots 8t + k up to
// B q (B <= 8); out, coefficients t + 256k up to 32q. buf as above, with the words
// 8t + k (own) free.
template <int P, uint32_t B = 5>
__device__ __forceinline__ void nr_inverse(uint32_t (&x)[P][8], uint32_t (*buf)[POLY4_LDS], const nr_u32x2* tw,
                                           uint32_t t, const NrLimb& m) {
    NrTw w;
    nr_tw_load(w, tw, nr_inv_node(3, t), false);
    nr_inv_phase<P, false, B>(x, w, m);  // sums of four: 4B q at k = 0 and 4, else up to 4q
#pragma unroll
    for (int p = 0; p < P; p++) {
        x[p][0] = nr_reduce(x[p][0], m);
        x[p][4] = nr_reduce(x[p][4], m);
    }
    nr_store<3, P>(buf, x, t);
    nr_tw_load(w, tw, nr_inv_node(2, t), true);
    lds_barrier();
    nr_load<2, P>(buf, x, t);
    nr_inv_phase<P, true, 4>(x, w, m);  // 32q at k = 0, 8q at k = 1, else up to 4q
#pragma unroll
    for (int p = 0; p < P; p++) {
        x[p][0] = nr_reduce(x[p][0], m);
        x[p][1] = nr_reduce(x[p][1], m);
    }
    nr_store<2, P>(buf, x, t);
    nr_tw_load(w, tw, nr_inv_node(1, t), true);
    lds_barrier();
    nr_load<1, P>(buf, x, t);
    nr_inv_phase<P, true, 4>(x, w, m);
#pragma unroll
    for (int p = 0; p < P; p++) {
        x[p][0] = nr_reduce(x[p][0], m);
        x[p][1] = nr_reduce(x[p][1], m);
    }
    nr_store<1, P>(buf, x, t);
    nr_tw_load(w, tw, nr_inv_node(0, t), true);
    lds_barrier();
    nr_load<0, P>(buf, x, t);
    nr_inv_phase<P, true, 4>(x, w, m);
}

// Both limbs' forward tables as (w, companion) pairs in LDS ([limb][N]);
// the caller synchronises.
__device__ __forceinline__ void nr_stage_twiddles(nr_u32x2 (*tw)[N], const NttConst& nc, uint32_t tid,
                                                  uint32_t nthreads) {
    for (uint32_t x = tid; x < 2 * N; x += nthreads) {
        const uint32_t limb = x / N, i = x % N;
        const uint32_t* b = nc.tw + (size_t)limb * 4 * N;
        tw[limb][i] = nr_u32x2{b[i], b[N + i]};
    }
}

// Gadget constants: the inverse transform's N^-1 and the CRT lift's cofactor
// inverse in one Shoup factor per limb.
struct NrGadget {
    uint32_t k[2], kp[2];
};
inline NrGadget nr_gadget_const(const NttConst& nc, const CrtConst& cc) {
    NrGadget g;
    for (int c = 0; c < 2; c++) {
        const uint64_t q = qof(c);
        g.k[c] = (uint32_t)((uint64_t)nc.inv_n[c] * (c ? cc.q0inv_q1 : cc.q1inv_q0) % q);
        g.kp[c] = (uint32_t)(((uint64_t)g.k[c] << 32) / q);
    }
    return g;
}
// One limb's share of the CRT lift from an unscaled inverse transform's
// output: t_c in [0, q_c) for limb 1, centred (|t_0| < q_0/2) for limb 0.
__device__ __forceinline__ uint32_t nr_crt_part(uint32_t x, const NrGadget& g, int c, const NrLimb& m) {
    const uint32_t r = fold(nr_mul(x, g.k[c], g.kp[c], m), m.q);
    const uint32_t h = c ? 0xffffffffu : Q0 / 2;
    return r > h ? r - m.q : r;
}
// Digits 1 and 2 of the centred lift (gadget2's): d1 as its 18 bits plus
// 2^17, d2 signed. v = t0 Q1 + t1 Q0 lies in (-Q/2, 3Q/2), so one
// subtraction centres it; adding 2^17 and 2^35 first makes both roundings
// plain shifts.
__device__ __forceinline__ nr_u32x2 nr_digits(uint32_t t0, uint32_t t1) {
    constexpr int64_t off = ((int64_t)1 << 17) + ((int64_t)1 << 35);
    int64_t v = (int64_t)(int32_t)t0 * (int32_t)Q1 + off;
    v = (int64_t)(int32_t)t1 * (int32_t)Q0 + v;
    v = v > (int64_t)(QFULL >> 1) + off ? v - (int64_t)QFULL : v;
    return nr_u32x2{(uint32_t)((uint64_t)v >> 18) & 0x3ffffu, (uint32_t)(int32_t)(v >> 36)};
}

// sum/2^32 mod q, below sum/2^32 + q, for sum < 2^63 (Montgomery).
__device__ __forceinline__ uint32_t nr_montgomery(uint64_t s, uint32_t qneg, uint32_t q) {
    const uint32_t k = (uint32_t)s * qneg;
    return (uint32_t)((s + (uint64_t)k * q) >> 32);
}
constexpr uint32_t nr_neg_inverse(uint32_t q) {  // -q^-1 mod 2^32
    uint32_t x = 1;
    for (int i = 0; i < 5; i++) x *= 2 - q * x;
    return 0u - x;
}

}  // namespace ipx
