// Horner chain split over two workgroups per chain, one per RNS limb.
//
// The step acc <- ext_prod(rgsw, acc) + packed[i] (reference
// src/gpu_online.cu:474-540, src/crypto.cpp:219-279) costs 4 INTTs, two
// gadget decompositions and 8 NTTs. Only the decomposition couples the
// limbs (its CRT lift needs both residues of a coefficient), so each limb's
// workgroup inverts its own two polynomials, swaps its shares of the lift
// with its partner through global memory, cuts every coefficient into
// digits itself and transforms the four digit polynomials mod its own
// prime: 6 transforms per workgroup and one exchange per step instead of 12
// transforms in one workgroup. Inside a workgroup, team p of 256 lanes has
// part p (a or b) of the accumulator: its inverse transform, its digits and
// their products with the query's rows; the teams add each other's half of
// the products through LDS. Transforms and layouts as in ntt_regs.h.
//
// Bound: like the one-workgroup chain, VALU issue of a serial chain, here on
// two CUs (about 4.3 us of a step), plus the exchange's latency (about 1.6).
// A step takes 5.9 us against the one workgroup's 8.6 (63 steps, one chain:
// 376 and 541 us); with transforms through LDS, and flags behind L2
// write-backs for the exchange, it took 12.
//
// Pairing: block b serves chain (b/16)*8 + b%8, limb (b/8)%2, so partners
// are b and b^8 (consecutive workgroups are spread over the XCDs
// round-robin, which puts partners on the same XCD). The exchange has no
// flag: a share takes 27 bits of a word, and the 5 upper bits of two words
// stored together (agent_store2, an 8-byte access, so they arrive together)
// hold the step's number; the partner loads them until the number is
// there. Against a counter behind the data that saves the wait for the
// stores and one trip through memory per step, and correctness depends on
// neither placement nor caches. Steps alternate between two buffers: a
// workgroup stores step n + 2 only after all of its lanes have seen the
// partner's step n + 1, which the partner's lanes store after they have read
// step n. The words must hold no number of this chain's steps beforehand
// (they are zeroed in the answer's preparation launch).
// The wait is bounded: a workgroup whose wait exceeds the bound (its partner
// has not had a CU for that long) sets *status and makes the whole chain, from
// its highest group, by itself: both limbs' polynomials in turn through the
// same buffers, the twiddles staged anew for each. It writes its own limb
// only, as ever, so its partner, whose wait then ends the same way, may run
// at any time. (The kernel takes 176 VGPRs with that path and 158 without:
// one workgroup to a CU either way.)
// With a bound of zero (to see chains give up) a workgroup fills its limb of
// the response with all-ones words instead (no residue; where the chain
// continues in a later launch, of the state, which passes them on).
#include "kernels.h"
#include "ntt_regs.h"

namespace ipx {

namespace {

constexpr size_t BLK = (size_t)D_EFF * 2 * N;
constexpr uint32_t kShareMask = (1u << 27) - 1, kShareCentre = 1u << 26;
static_assert(Q1 <= kShareMask && Q0 / 2 < kShareCentre, "a share fits 27 bits");

__global__ __launch_bounds__(256) void k_fill_u32(uint32_t* __restrict__ p, size_t n, uint32_t v) {
    for (size_t x = (size_t)blockIdx.x * 256 + threadIdx.x; x < n; x += (size_t)gridDim.x * 256) p[x] = v;
}

__global__ __launch_bounds__(512, 2) void k_horner_pair(const uint32_t* __restrict__ pa_base, size_t pa_stride,
                                                        uint32_t G, uint32_t Da, uint32_t T,
                                                        const uint32_t* __restrict__ packed_b, size_t pstride,
                                                        const uint32_t* __restrict__ rgsw, size_t rstride,
                                                        uint64_t* __restrict__ out, uint32_t* __restrict__ hstate,
                                                        uint32_t g_lo, uint32_t g_hi, uint32_t* xbuf,
                                                        uint32_t* status, uint32_t nchains, uint32_t spin_limit,
                                                        NttConst nc, NrGadget gc) {
    __shared__ __align__(16) uint32_t buf[2][2][POLY4_LDS];  // [team][digit polynomial]
    __shared__ __align__(16) nr_u32x2 tw[N];
    __shared__ uint32_t sx[2][8][256];  // products by the team that made them, for the other's part
    __shared__ uint32_t abort_flag;
    const uint32_t b = blockIdx.x, chain = (b >> 4) * 8 + (b & 7);
    const int c = (int)((b >> 3) & 1);
    if (chain >= nchains) return;  // both partners of a padding chain leave
    const uint32_t ct = chain % T, qi = chain / T, tid = threadIdx.x, t = tid & 255;
    const uint32_t p = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid >> 8));  // this team's part
    const uint32_t start = ct * Da;
    const uint32_t L = (G - start) < Da ? (G - start) : Da;
    const uint32_t top = start + L - 1;
    // this launch covers the chain's groups in [lo, hi), highest first
    const uint32_t lo = start > g_lo ? start : g_lo, hi = start + L < g_hi ? start + L : g_hi;
    if (lo >= hi) return;  // both partners leave
    const NrLimb m = nr_limb(c);
    // this team's part of a group: 8 consecutive slots of the limb
    auto load8 = [&](uint32_t (&x)[8], const uint32_t* src) {
        const nr_u32x4* s = reinterpret_cast<const nr_u32x4*>(src + (size_t)c * N + 8 * t);
        const nr_u32x4 l = s[0], u = s[1];
#pragma unroll
        for (int k = 0; k < 4; k++) {
            x[k] = l[k];
            x[k + 4] = u[k];
        }
    };
    const uint32_t* pk = p ? packed_b + qi * pstride : pa_base;
    const size_t pk_stride = p ? 2 * (size_t)N : pa_stride;
    uint32_t* hs = hstate + ((size_t)qi * T + ct) * 4 * N;  // chain state between launches, [a|b][limb][N]
    uint64_t* o = out + ((size_t)qi * T + ct) * 4 * N;
    auto give_up = [&]() {
        if (lo > start) {
            nr_u32x4* d = reinterpret_cast<nr_u32x4*>(hs + ((size_t)2 * p + c) * N + 8 * t);
            d[0] = d[1] = nr_u32x4{~0u, ~0u, ~0u, ~0u};
            return;
        }
        for (int k = 0; k < 8; k++) o[((size_t)2 * p + c) * N + t + 256 * k] = ~0ull;
    };
    uint32_t acc[1][8];  // slots 8t + k
    int first;
    bool alone = false;
    if (top < g_hi) {  // the chain starts here: acc = packed[top]
        load8(acc[0], pk + (size_t)top * pk_stride);
        first = (int)top - 1;
    } else {
        load8(acc[0], hs + (size_t)p * 2 * N);
        first = (int)hi - 1;
        if (acc[0][0] == ~0u) {  // every lane: the chain gave up in an earlier launch
            give_up();
            return;
        }
    }
    if (first >= (int)lo) {
        for (uint32_t x = tid; x < N; x += 512) {  // published by the barrier below
            const uint32_t* f = nc.tw + (size_t)c * 4 * N;
            tw[x] = nr_u32x2{f[x], f[N + x]};
        }
        if (tid == 0) abort_flag = 0;
        // the query's rows for this part's digits [to a | to b][digit][slot], times 2^32 mod q
        const uint32_t r32 = c ? (uint32_t)(4294967296ull % Q1) : (uint32_t)(4294967296ull % Q0);
        const uint32_t qneg = c ? nr_neg_inverse(Q1) : nr_neg_inverse(Q0);
        const uint32_t* rg = rgsw + qi * rstride + (size_t)2 * p * BLK;
        uint32_t rows[2][2][8];
#pragma unroll
        for (int r = 0; r < 2; r++)
#pragma unroll
            for (int j = 0; j < 2; j++) {
                load8(rows[r][j], rg + (size_t)r * BLK + (size_t)j * 2 * N);
#pragma unroll
                for (int k = 0; k < 8; k++) rows[r][j][k] = mul_mod(rows[r][j][k], r32, c);
            }
        // [parity][limb][part][k/2][lane][2]
        uint32_t* xw = xbuf + (size_t)chain * 8 * N + ((size_t)c * 2 + p) * N + 2 * t;
        const uint32_t* xr = xbuf + (size_t)chain * 8 * N + ((size_t)(1 - c) * 2 + p) * N + 2 * t;
        __syncthreads();
        for (int gs = first; gs >= (int)lo; gs--) {
            const uint32_t step = top - (uint32_t)gs;  // 1, 2, ...
            const uint32_t par = (step & 1) * 4 * N;
            // 1..1023: 5 bits in each of the two words of an access
            const uint32_t num = (step - 1) % 1023 + 1, tag0 = num << 27, tag1 = (num >> 5) << 27;
            uint32_t cf[1][8];  // coefficients t + 256k
#pragma unroll
            for (int k = 0; k < 8; k++) cf[0][k] = acc[0][k];
            nr_inverse<1, 6>(cf, buf[p], tw, t, m);
#pragma unroll
            for (int k = 0; k < 8; k++) cf[0][k] = nr_crt_part(cf[0][k], gc, c, m);
            const uint32_t off = c ? 0 : kShareCentre;
#pragma unroll
            for (int k = 0; k < 4; k++)
                agent_store2(xw + par + 512 * k, (cf[0][2 * k] + off) | tag0, (cf[0][2 * k + 1] + off) | tag1);
            uint32_t pv[8];  // the step's packed part, in flight during the exchange
            load8(pv, pk + (size_t)gs * pk_stride);
            uint32_t other[8];
            uint32_t spins = 0;
            bool late = spin_limit == 0;
            while (!late) {
                uint32_t diff = 0;
#pragma unroll
                for (int k = 0; k < 4; k++) {
                    const uint64_t v = agent_load2(xr + par + 512 * k);
                    other[2 * k] = (uint32_t)v;
                    other[2 * k + 1] = (uint32_t)(v >> 32);
                    diff |= (other[2 * k] ^ tag0) | (other[2 * k + 1] ^ tag1);
                }
                if (diff <= kShareMask) break;
                late = ++spins > spin_limit;
            }
            if (late) {
                __hip_atomic_store(status, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                abort_flag = 1;
            }
            lds_barrier();
            if (abort_flag) {
                if (spin_limit == 0) {
                    give_up();
                    return;
                }
                alone = true;
                break;
            }
            uint32_t x[2][8];  // digit polynomials: residues + q mod this limb's prime
#pragma unroll
            for (int k = 0; k < 8; k++) {
                const uint32_t got = (other[k] & kShareMask) - (c ? kShareCentre : 0);
                const nr_u32x2 d = nr_digits(c ? got : cf[0][k], c ? cf[0][k] : got);
                x[0][k] = d.x + (m.q - (1u << 17));
                x[1][k] = d.y + m.q;
            }
            nr_forward<2>(x, buf[p], tw, t, m, [] { lds_barrier(); });
            uint32_t mine[8];
#pragma unroll
            for (int k = 0; k < 8; k++) {
                // digits below 23.1q, rows below q: the sums stay below 47 q^2, a product below 2.1q
                uint64_t s[2];
#pragma unroll
                for (int r = 0; r < 2; r++)
                    s[r] = (uint64_t)x[0][k] * rows[r][0][k] + (uint64_t)x[1][k] * rows[r][1][k];
                mine[k] = nr_montgomery(p ? s[1] : s[0], qneg, m.q);
                sx[p][k][t] = nr_montgomery(p ? s[0] : s[1], qneg, m.q);
            }
            lds_barrier();
#pragma unroll
            for (int k = 0; k < 8; k++) acc[0][k] = mine[k] + sx[1 - p][k][t] + pv[k];  // below 5.2q
        }
        if (alone) {
            // this team's part of both limbs, canonical between steps
            uint32_t a0[8], a1[8];
            auto load_limb = [&](uint32_t (&x)[8], const uint32_t* src, int l) {
#pragma unroll
                for (int k = 0; k < 8; k++) x[k] = src[(size_t)l * N + 8 * t + k];
            };
            load_limb(a0, pk + (size_t)top * pk_stride, 0);
            load_limb(a1, pk + (size_t)top * pk_stride, 1);
#pragma unroll 1
            for (int gs = (int)top - 1; gs >= (int)lo; gs--) {
                uint32_t s0[8] = {}, s1[8] = {};  // shares of the lift, then the digits
#pragma unroll 1
                for (int half = 0; half < 4; half++) {  // inverse of limb 0, 1, then products mod limb 0, 1
                    const int l = half & 1;
                    const NrLimb ml = nr_limb(l);
                    __syncthreads();  // the last transform's twiddles and products are read
                    for (uint32_t x = tid; x < N; x += 512) {
                        const uint32_t* f = nc.tw + (size_t)l * 4 * N;
                        tw[x] = nr_u32x2{f[x], f[N + x]};
                    }
                    __syncthreads();
                    if (half < 2) {
                        uint32_t cf[1][8];
#pragma unroll
                        for (int k = 0; k < 8; k++) cf[0][k] = l ? a1[k] : a0[k];
                        nr_inverse<1, 6>(cf, buf[p], tw, t, ml);
#pragma unroll
                        for (int k = 0; k < 8; k++) {
                            const uint32_t v = nr_crt_part(cf[0][k], gc, l, ml);
                            s0[k] = l ? s0[k] : v;
                            s1[k] = l ? v : s1[k];
                        }
                        if (half == 0) continue;
#pragma unroll
                        for (int k = 0; k < 8; k++) {
                            const nr_u32x2 d = nr_digits(s0[k], s1[k]);
                            s0[k] = d.x;
                            s1[k] = d.y;
                        }
                        continue;
                    }
                    uint32_t x[2][8];
#pragma unroll
                    for (int k = 0; k < 8; k++) {
                        x[0][k] = s0[k] + (ml.q - (1u << 17));
                        x[1][k] = s1[k] + ml.q;
                    }
                    nr_forward<2>(x, buf[p], tw, t, ml, [] { lds_barrier(); });
                    uint32_t pv[8];
                    load_limb(pv, pk + (size_t)gs * pk_stride, l);
#pragma unroll
                    for (int k = 0; k < 8; k++) {
#pragma unroll
                        for (int j = 0; j < 2; j++) x[j][k] = fold(nr_reduce(x[j][k], ml), ml.q);
                        const uint32_t* r = rg + (size_t)l * N + 8 * t + k;
                        const uint32_t ta = red64((uint64_t)x[0][k] * r[0] + (uint64_t)x[1][k] * r[2 * N], l);
                        const uint32_t tb = red64((uint64_t)x[0][k] * r[BLK] + (uint64_t)x[1][k] * r[BLK + 2 * N], l);
                        pv[k] = add_mod(pv[k], p ? tb : ta, ml.q);
                        sx[p][k][t] = p ? ta : tb;
                    }
                    __syncthreads();
#pragma unroll
                    for (int k = 0; k < 8; k++) {
                        const uint32_t v = add_mod(pv[k], sx[1 - p][k][t], ml.q);
                        a0[k] = l ? a0[k] : v;
                        a1[k] = l ? v : a1[k];
                    }
                }
            }
#pragma unroll
            for (int k = 0; k < 8; k++) acc[0][k] = c ? a1[k] : a0[k];
        }
#pragma unroll
        for (int k = 0; k < 8; k++) acc[0][k] = fold(fold(fold(acc[0][k], 4 * m.q), 2 * m.q), m.q);
    }
    if (lo > start) {  // the chain continues in a later launch
        nr_u32x4* d = reinterpret_cast<nr_u32x4*>(hs + ((size_t)2 * p + c) * N + 8 * t);
        d[0] = nr_u32x4{acc[0][0], acc[0][1], acc[0][2], acc[0][3]};
        d[1] = nr_u32x4{acc[0][4], acc[0][5], acc[0][6], acc[0][7]};
        return;
    }
    // the response, through LDS for whole lines of 8-byte words (a lane's own
    // words of the last exchange)
    nr_store<3, 1>(buf[p], acc, t);
    __syncthreads();
#pragma unroll
    for (int k = 0; k < 8; k++)
        o[((size_t)2 * p + c) * N + t + 256 * k] = buf[p][0][nr_base(0, t) + nr_stride<0>() * k];
}

}  // namespace

size_t horner_pair_xbuf_words(size_t nchains) { return nchains * 2 * 2 * 2 * N; }

hipError_t launch_horner_pair(const uint32_t* pa_base, size_t pa_stride, size_t G, size_t Da, size_t T,
                              const uint32_t* packed_b, size_t packed_stride, const uint32_t* rgsw,
                              size_t rgsw_stride, uint64_t* out, uint32_t* hstate, size_t g_lo, size_t g_hi,
                              size_t nq, uint32_t* xbuf, uint32_t* status, uint32_t spin_limit, const NttConst& nc,
                              const CrtConst& cc, hipStream_t s) {
    const size_t nchains = nq * T;
    if (nchains == 0 || g_lo >= g_hi) return hipSuccess;
    const size_t blocks = 16 * ((nchains + 7) / 8);
    hipLaunchKernelGGL(k_horner_pair, dim3((unsigned)blocks), dim3(512), 0, s, pa_base, pa_stride, (uint32_t)G,
                       (uint32_t)Da, (uint32_t)T, packed_b, packed_stride, rgsw, rgsw_stride, out, hstate,
                       (uint32_t)g_lo, (uint32_t)g_hi, xbuf, status, (uint32_t)nchains, spin_limit, nc,
                       nr_gadget_const(nc, cc));
    return hipGetLastError();
}

hipError_t launch_fill_u32(uint32_t* p, size_t n, uint32_t v, hipStream_t s) {
    if (n == 0) return hipSuccess;
    size_t blocks = (n + 255) / 256;
    if (blocks > 1024) blocks = 1024;
    hipLaunchKernelGGL(k_fill_u32, dim3((unsigned)blocks), dim3(256), 0, s, p, n, v);
    return hipGetLastError();
}

}  // namespace ipx
