// One-time preprocessing kernels for gfx950: in-place encode (inverse DFT
// over Z_P[X]/(X^N+1)), the a-side matmul, the ring embedding and the
// CollapseA chains that produce the per-group precomp tensors.
//
// Semantics follow the reference preprocess (src/gpu_protocol.cu:535-817):
// encode (src/gpu_preprocess.cu:931-1034), a32 = N^-1 * reversed
// sum_r NTT(db column slice) * NTT(tau_{2N-1}(a_r))
// (src/gpu_preprocess.cu:347-410), ring embed + automorphism
// (src/gpu_preprocess.cu:39-92, :158-194), collapse (src/gpu_preprocess.cu:
// 452-881). Two re-formulations replace the reference's kernels while
// producing the same values:
//  * ring embed: the 2^34-MAC sum per group is the evaluation of
//    P_{c,p}(Y) = sum_j a32[j][c][p] Y^j at the odd powers of psi, i.e. a
//    length-N negacyclic NTT along j; combined with the automorphism
//    permutation, a_post[k][c][i] = F[c][perm_{+-5^k}(i)][i] with
//    F[c][p] = NTT(a32[.][c][p]).
//  * encode: the transform factors by coefficient residue k mod (2N/D) into
//    independent D x D/2 negacyclic blocks, each done in LDS in one pass
//    over the DB instead of log2(D)+2 global passes.
#include "kernels.h"
#include "ntt_regs.h"

namespace ipx {

namespace {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ uint32_t modp(uint32_t x) {  // x mod 65535, any u32
    uint32_t r = (x & 0xffffu) + (x >> 16);
    r = (r & 0xffffu) + (r >> 16);
    return r >= PMOD ? r - PMOD : r;
}

// ------------------------------------------------------------ encode
// Block (row, ct, k0-chunk). Sub-problem for residue k0 of the coefficient
// index mod S = 2N/Da: y[d][k1] = x[d][k0 + S*k1], k1 < Da/2, on which
// X^S acts as a negacyclic shift. out[m] = Da^-1 sum_d y[d] * X^(-2N d m/Da)
// computed as a radix-2 DIT FFT (bit-reversed load, natural-order output).
// Bound: index arithmetic and LDS; every extent is a power of two, given by
// its logarithm, and consecutive lanes take consecutive k0 (then k1), hence
// consecutive LDS words. With divisions by the extents and k0 outermost
// (64-byte strides between lanes) 1 GB took 3.3 ms, now 2.1. The chunks of one
// row share cache lines: workgroup numbers 8 apart, one XCD, hold them.
__global__ __launch_bounds__(1024) void k_encode(uint16_t* __restrict__ db, uint32_t C, uint32_t T, uint32_t lda,
                                                 uint32_t lkc, uint32_t lch, uint32_t Dinv) {
    __shared__ uint16_t y[32768];  // [d][k1][k0]
    const uint32_t idx = blockIdx.x >> 3, unit = ((idx >> lch) << 3) + (blockIdx.x & 7);
    const uint32_t row = unit / T, ct = unit % T, chunk = idx & ((1u << lch) - 1);
    const uint32_t l1 = lda - 1, S = 2 * N >> lda, L1 = 1u << l1, lrow = l1 + lkc, E = 1u << (lda + lrow);
    const uint32_t mk = (1u << lkc) - 1, m1 = L1 - 1;
    uint16_t* base = db + (size_t)row * C + (((size_t)ct * N) << lda) + ((size_t)chunk << lkc);
    for (uint32_t x = threadIdx.x; x < E; x += 1024) {
        const uint32_t k0 = x & mk, k1 = (x >> lkc) & m1, d = x >> lrow;
        const uint32_t dr = __builtin_bitreverse32(d) >> (32 - lda);
        y[(dr << lrow) + (x & ((1u << lrow) - 1))] = base[(size_t)d * N + S * k1 + k0];
    }
    __syncthreads();
    const uint32_t npairs = E / 2;
    for (uint32_t lv = 0; lv < lda; lv++) {
        const uint32_t half = 1u << lv;
        uint16_t sum[16], dif[16];
#pragma unroll
        for (int r = 0; r < 16; r++) {
            const uint32_t z = threadIdx.x + 1024 * r;
            if (z < npairs) {
                const uint32_t k0 = z & mk, k1 = (z >> lkc) & m1, pidx = z >> lrow, ph = pidx & (half - 1);
                const uint32_t de = ((pidx >> lv) << (lv + 1)) + ph, dodd = de + half;
                const uint32_t src = k1 + (ph << (lda - lv - 1));
                const uint32_t e = y[(de << lrow) + (k1 << lkc) + k0];
                uint32_t o = y[(dodd << lrow) + ((src & m1) << lkc) + k0];
                if (src >= L1 && o) o = PMOD - o;
                uint32_t a = e + o;
                if (a >= PMOD) a -= PMOD;
                uint32_t b = e + PMOD - o;
                if (b >= PMOD) b -= PMOD;
                sum[r] = (uint16_t)a;
                dif[r] = (uint16_t)b;
            }
        }
        __syncthreads();
#pragma unroll
        for (int r = 0; r < 16; r++) {
            const uint32_t z = threadIdx.x + 1024 * r;
            if (z < npairs) {
                const uint32_t pidx = z >> lrow, in = z & ((1u << lrow) - 1);
                const uint32_t de = ((pidx >> lv) << (lv + 1)) + (pidx & (half - 1)), dodd = de + half;
                y[(de << lrow) + in] = sum[r];
                y[(dodd << lrow) + in] = dif[r];
            }
        }
        __syncthreads();
    }
    for (uint32_t x = threadIdx.x; x < E; x += 1024) {
        const uint32_t k0 = x & mk, k1 = (x >> lkc) & m1, d = x >> lrow;
        base[(size_t)d * N + S * k1 + k0] = (uint16_t)modp((uint32_t)y[x] * Dinv);
    }
}

// ------------------------------------------------------------ a-side
// Block (group, 4 columns) over the resident DB (byte planes in 16-row
// blocks): acc[col][c] = sum_r NTT(db[rN..rN+N-1][col]) * crs[r][c]; a32T[g][c][k][col] = N^-1 * acc[col][c][N-1-k].
// Team c of 256 lanes transforms the 4 columns mod its limb's prime in
// registers (ntt_regs.h) and keeps 8 slots of each sum. The columns' units
// (one per lane and plane, the next polynomial's in flight during the
// transforms) become 16-bit values in LDS, which both teams read. Products
// (below 23q * q < 2^58) add up in 64 bits, reduced every 32 polynomials.
// Bound: VALU issue. With every transform through LDS and byte loads (1024
// lanes, two polynomials per team) 1 GB took 3.7 ms, now 1.6.
__global__ __launch_bounds__(512, 2) void k_aside(const uint8_t* __restrict__ db, uint32_t C, uint32_t nr, uint32_t g0,
                                                  const uint32_t* __restrict__ crs, uint32_t* __restrict__ a32T,
                                                  NttConst nc) {
    __shared__ __align__(16) uint32_t buf[2][4][POLY4_LDS];
    __shared__ __align__(16) nr_u32x2 tw2[2][N];
    __shared__ __align__(16) uint16_t xin[4][N + 16];
    const uint32_t gl = blockIdx.x / (N / 4), j0 = (blockIdx.x % (N / 4)) * 4;
    const uint32_t tid = threadIdx.x, t = tid & 255;
    const int c = __builtin_amdgcn_readfirstlane((int)(tid >> 8));
    const NrLimb m = nr_limb(c);
    nr_stage_twiddles(tw2, nc, tid, 512);  // published by the first barrier below
    const uint32_t kb = tid >> 2, col = tid & 3;  // this lane's unit
    const u32x4* src = reinterpret_cast<const u32x4*>(db) + (size_t)kb * 2 * C + (size_t)(g0 + gl) * N + j0 + col;
    const size_t rstep = (size_t)(N / 16) * 2 * C;
    u32x4 lo = src[0], hi = src[C];
    uint64_t acc[4][8];
#pragma unroll
    for (int p = 0; p < 4; p++)
#pragma unroll
        for (int k = 0; k < 8; k++) acc[p][k] = 0;
    for (uint32_t r = 0; r < nr; r++) {
        // the transforms' barriers below keep this behind the last reads
        u32x4* d = reinterpret_cast<u32x4*>(&xin[col][16 * kb]);
        u32x4 v[2];
#pragma unroll
        for (int w = 0; w < 4; w++) {
            v[w >> 1][2 * (w & 1)] = __builtin_amdgcn_perm(hi[w], lo[w], 0x05010400u);
            v[w >> 1][2 * (w & 1) + 1] = __builtin_amdgcn_perm(hi[w], lo[w], 0x07030602u);
        }
        d[0] = v[0];
        d[1] = v[1];
        lds_barrier();
        if (r + 1 < nr) {
            lo = src[(r + 1) * rstep];
            hi = src[(r + 1) * rstep + C];
        }
        const u32x4* A = reinterpret_cast<const u32x4*>(crs + ((size_t)r * 2 + c) * N + 8 * t);
        const u32x4 a0 = A[0], a1 = A[1];
        uint32_t x[4][8];
#pragma unroll
        for (int p = 0; p < 4; p++)
#pragma unroll
            for (int k = 0; k < 8; k++) x[p][k] = xin[p][t + 256 * k];
        nr_forward<4>(x, buf[c], tw2[c], t, m, [] { lds_barrier(); });
#pragma unroll
        for (int p = 0; p < 4; p++)
#pragma unroll
            for (int k = 0; k < 8; k++) acc[p][k] += (uint64_t)x[p][k] * (k < 4 ? a0[k & 3] : a1[k & 3]);
        if ((r & 31) == 31) {
#pragma unroll
            for (int p = 0; p < 4; p++)
#pragma unroll
                for (int k = 0; k < 8; k++) acc[p][k] = red64(acc[p][k], c);
        }
    }
#pragma unroll
    for (int k = 0; k < 8; k++) {
        uint32_t o[4];
#pragma unroll
        for (int p = 0; p < 4; p++) o[p] = mul_shoup(red64(acc[p][k], c), nc.inv_n[c], nc.inv_n_p[c], m.q);
        *reinterpret_cast<u32x4*>(a32T + (((size_t)gl * 2 + c) * N + (N - 1 - (8 * t + k))) * N + j0) =
            u32x4{o[0], o[1], o[2], o[3]};
    }
}

// ------------------------------------------------------------ ring embed
// In-place forward NTT of a32T rows; row x = (g*2 + c)*N + p has limb c.
__global__ __launch_bounds__(256) void k_ntt_rows(uint32_t* __restrict__ rows, NttConst nc) {
    __shared__ uint32_t buf[POLY_LDS];
    const int limb = (int)((blockIdx.x >> LOGN) & 1);
    uint32_t* p = rows + (size_t)blockIdx.x * N;
    const uint32_t t = threadIdx.x;
#pragma unroll
    for (int k = 0; k < 8; k++) buf[ls(t + 256 * k)] = p[t + 256 * k];
    __syncthreads();
    ntt_fwd_lds(buf, t, tw_global(nc, limb), limb);
#pragma unroll
    for (int k = 0; k < 8; k++) p[t + 256 * k] = buf[ls(t + 256 * k)];
}

// ------------------------------------------------------------ a_post gather
// a_post of every step of both directions, F[c][p(s, i)][i], into the words
// where the chain's digit 0 of that step goes (dtmp [dir][c][s][0][i]): the
// chain then reads whole lines instead of one line per value. Block (group,
// limb, 16 slots i): the slots' 16 columns of F in LDS (128 KiB), read and
// written in 64-byte rows.
__global__ __launch_bounds__(1024) void k_apost_gather(const uint32_t* __restrict__ F, uint32_t* __restrict__ dtmp) {
    __shared__ __align__(16) uint32_t T[N][16];
    __shared__ uint16_t pw[NSTEPS];  // 5^(N/2-2-s) mod 2N
    const uint32_t it = blockIdx.x % (N / 16), c = (blockIdx.x / (N / 16)) & 1, gl = blockIdx.x / (2 * (N / 16));
    const uint32_t i0 = it * 16, tid = threadIdx.x;
    const uint32_t* Fg = F + ((size_t)gl * 2 + c) * N * N + i0;
    for (uint32_t x = tid; x < N * 4; x += 1024)
        *reinterpret_cast<u32x4*>(&T[x >> 2][4 * (x & 3)]) =
            *reinterpret_cast<const u32x4*>(Fg + (size_t)(x >> 2) * N + 4 * (x & 3));
    if (tid < NSTEPS) {
        uint32_t ts = 1;
        for (uint32_t ex = HALF - 2 - tid, b = 5; ex; ex >>= 1, b = (b * b) & (2 * N - 1))
            if (ex & 1) ts = (ts * b) & (2 * N - 1);
        pw[tid] = (uint16_t)ts;
    }
    __syncthreads();
    const uint32_t il = tid & 15, v = 2 * brev11(i0 + il) + 1;
    for (uint32_t r = tid >> 4; r < 2 * NSTEPS; r += 64) {
        const uint32_t dir = r >= NSTEPS, s = r - dir * NSTEPS;
        const uint32_t pf = perm_slot(pw[s], v), p = dir ? N - 1 - pf : pf;
        dtmp[((size_t)gl * 2 + dir) * RD_SZ + ((size_t)c * NSTEPS + s) * D_EFF * N + i0 + il] = T[p][il];
    }
}

// ------------------------------------------------------------ collapse
// One block per (group, direction): 1023 dependent steps. Step s folds
// k = N/2-1-s: state -> INTT -> gadget digits 1,2 -> NTT -> D[s]; state =
// a_post[k-1] - sum_j D[s][j] * K[j][perm]. Both the expanded key of step s
// (tau_{+-5^(k-1)} of ksk5a, reference kskstep = n_steps-1-s) and a_post[k-1]
// are gathered through the same slot permutation p; k_apost_gather has put
// the latter where the step's first digit will go.
// A serial chain on one CU, built like the Horner chain: a 256-lane team per
// limb keeps 8 slots of its polynomials in registers between transforms
// (ntt_regs.h), the teams swap halves of the CRT lift and the digits through
// LDS, and the key is kept times 2^32 for Montgomery products. Every
// transform through LDS by its own 256 lanes of 1024 took 13.3 us per step;
// with the a_post values gathered in the step (4 bytes of each of 4096 cache
// lines, the most a CU's misses allow) this form took 11.4.
__global__ __launch_bounds__(512, 2) void k_collapse_chain(const uint32_t* __restrict__ F,
                                                           const uint32_t* __restrict__ ksk5a,
                                                           uint32_t* dtmp,
                                                           uint32_t* __restrict__ states, NttConst nc, NrGadget gc) {
    __shared__ __align__(16) uint32_t buf[2][2][POLY4_LDS];
    __shared__ __align__(16) nr_u32x2 tw2[2][N];
    __shared__ uint32_t K[2][2][N];         // [limb][digit][slot], times 2^32 mod q
    __shared__ uint32_t xs[2][4][256];      // lift shares by the team that sent them
    __shared__ uint32_t dx[2][4][2][256];   // digits by the team that made them
    const uint32_t gl = blockIdx.x, dir = blockIdx.y, tid = threadIdx.x, t = tid & 255;
    const int c = __builtin_amdgcn_readfirstlane((int)(tid >> 8));
    const NrLimb m = nr_limb(c);
    const uint32_t r32 = c ? (uint32_t)(4294967296ull % Q1) : (uint32_t)(4294967296ull % Q0);
    const uint32_t qneg = c ? nr_neg_inverse(Q1) : nr_neg_inverse(Q0);
    nr_stage_twiddles(tw2, nc, tid, 512);
    for (uint32_t x = t; x < 2 * N; x += 256)  // ksk5a [digit][limb][N]
        K[c][x / N][x % N] = mul_mod(ksk5a[((size_t)(x / N) * 2 + c) * N + x % N], r32, c);
    const uint32_t* Fg = F + ((size_t)gl * 2 + c) * N * N;
    uint32_t* Dout = dtmp + ((size_t)gl * 2 + dir) * RD_SZ + (size_t)c * NSTEPS * D_EFF * N;
    const nr_u32x2* tw = tw2[c];
    // t = 5^(N/2-1) mod 2N, then 5^(N/2-2-s) for step s
    uint32_t ts = 1;
    for (uint32_t ex = HALF - 1, b = 5; ex; ex >>= 1, b = (b * b) & (2 * N - 1))
        if (ex & 1) ts = (ts * b) & (2 * N - 1);
    uint32_t v[8];  // 2 BR(slot) + 1 of this lane's slots 8t + k
#pragma unroll
    for (int k = 0; k < 8; k++) v[k] = 2 * brev11(8 * t + k) + 1;
    auto slot = [&](int k) {
        const uint32_t pf = perm_slot(ts, v[k]);
        return dir ? N - 1 - pf : pf;
    };
    uint32_t st[1][8];
#pragma unroll
    for (int k = 0; k < 8; k++) st[0][k] = Fg[(size_t)slot(k) * N + 8 * t + k];
    __syncthreads();
    for (uint32_t s = 0; s < NSTEPS; s++) {
        ts = (ts * 3277u) & (2 * N - 1);  // times 5^-1
        uint32_t p[8];
#pragma unroll
        for (int k = 0; k < 8; k++) p[k] = slot(k);
        u32x4* D0 = reinterpret_cast<u32x4*>(Dout + (size_t)s * D_EFF * N + 8 * t);
        const u32x4 nl = D0[0], nh = D0[1];  // this step's a_post, the lane's own words
        const uint32_t nxt[8] = {nl[0], nl[1], nl[2], nl[3], nh[0], nh[1], nh[2], nh[3]};
        nr_inverse<1>(st, buf[c], tw, t, m);
        // team c lifts the coefficients k in [4c, 4c + 4) and sends the others
        uint32_t keep[4];
#pragma unroll
        for (int k = 0; k < 8; k++) st[0][k] = nr_crt_part(st[0][k], gc, c, m);
#pragma unroll
        for (int k = 0; k < 4; k++) {
            keep[k] = c ? st[0][k + 4] : st[0][k];
            xs[c][k][t] = c ? st[0][k] : st[0][k + 4];
        }
        lds_barrier();
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const uint32_t other = xs[1 - c][k][t];
            const nr_u32x2 d = nr_digits(c ? other : keep[k], c ? keep[k] : other);
            dx[c][k][0][t] = d.x;
            dx[c][k][1][t] = d.y;
        }
        lds_barrier();
        uint32_t x[2][8];  // digit polynomials: residues + q mod this limb's prime
#pragma unroll
        for (int h = 0; h < 2; h++)
#pragma unroll
            for (int k = 0; k < 4; k++) {
                x[0][4 * h + k] = dx[h][k][0][t] + (m.q - (1u << 17));
                x[1][4 * h + k] = dx[h][k][1][t] + m.q;
            }
        nr_forward<2>(x, buf[c], tw, t, m, [] { lds_barrier(); });
#pragma unroll
        for (int j = 0; j < 2; j++) {
#pragma unroll
            for (int k = 0; k < 8; k++) x[j][k] = fold(nr_reduce(x[j][k], m), m.q);  // canonical, from at most 24q
            u32x4* d = D0 + j * (N / 4);
            d[0] = u32x4{x[j][0], x[j][1], x[j][2], x[j][3]};
            d[1] = u32x4{x[j][4], x[j][5], x[j][6], x[j][7]};
        }
#pragma unroll
        for (int k = 0; k < 8; k++) {
            const uint64_t acc = (uint64_t)x[0][k] * K[c][0][p[k]] + (uint64_t)x[1][k] * K[c][1][p[k]];
            st[0][k] = nxt[k] + (2 * m.q - nr_montgomery(acc, qneg, m.q));  // the product below 1.1q: st below 3q
        }
    }
#pragma unroll
    for (int k = 0; k < 8; k++)
        states[(((size_t)gl * 2 + dir) * 2 + c) * N + 8 * t + k] = fold(fold(st[0][k], 2 * m.q), m.q);
}

// Final CollapseOne: digits of the conjugate chain's last state -> D_final;
// a = (forward chain's last state) - sum_j D_final[j] * NTT(ksk_neg1 a-part)[j].
__global__ __launch_bounds__(1024) void k_collapse_final(const uint32_t* __restrict__ states,
                                                         const uint32_t* __restrict__ kneg1a,
                                                         uint32_t* __restrict__ precomp_g0, NttConst nc,
                                                         CrtConst cc) {
    __shared__ uint32_t buf[4][POLY_LDS];
    __shared__ uint32_t twl[8 * N];
    const uint32_t gl = blockIdx.x, tid = threadIdx.x, team = tid >> 8, t = tid & 255;
    stage_twiddles(twl, nc, tid, 1024);
    const int tlimb = (int)(team & 1);
    const Tw tw = tw_lds(twl, tlimb);
    const uint32_t* sf = states + (size_t)gl * 4 * N;  // dir 0
    const uint32_t* sc = sf + 2 * N;                   // dir 1
    uint32_t* pc = precomp_g0 + (size_t)gl * PC_GROUP;
#pragma unroll
    for (int e = 0; e < 2; e++) {
        buf[0][ls(tid + 1024 * e)] = sc[tid + 1024 * e];
        buf[1][ls(tid + 1024 * e)] = sc[N + tid + 1024 * e];
    }
    __syncthreads();
    ntt_inv_lds(buf[team], t, tw, tlimb, nc.inv_n[tlimb], nc.inv_n_p[tlimb], team < 2);
    uint32_t d0[2][2], d1[2][2];
#pragma unroll
    for (int e = 0; e < 2; e++) gadget2(buf[0][ls(tid + 1024 * e)], buf[1][ls(tid + 1024 * e)], cc, d0[e], d1[e]);
    __syncthreads();
#pragma unroll
    for (int e = 0; e < 2; e++)
#pragma unroll
        for (int j = 0; j < 2; j++) {
            buf[j * 2 + 0][ls(tid + 1024 * e)] = d0[e][j];
            buf[j * 2 + 1][ls(tid + 1024 * e)] = d1[e][j];
        }
    __syncthreads();
    ntt_fwd_lds(buf[team], t, tw, tlimb);
#pragma unroll
    for (int c = 0; c < 2; c++)
#pragma unroll
        for (int e = 0; e < 2; e++) {
            const uint32_t i = tid + 1024 * e;
            uint64_t acc = 0;
#pragma unroll
            for (int j = 0; j < 2; j++) {
                const uint32_t dv = buf[j * 2 + c][ls(i)];
                pc[PC_DF + ((size_t)c * D_EFF + j) * N + i] = dv;
                acc += (uint64_t)dv * kneg1a[((size_t)j * 2 + c) * N + i];
            }
            pc[PC_A + (size_t)c * N + i] = sub_mod(sf[(size_t)c * N + i], red64(acc, c), qof(c));
        }
}

}  // namespace

hipError_t launch_encode(uint16_t* db, size_t R, size_t C, size_t Da, hipStream_t s) {
    if (Da <= 1) return hipSuccess;
    uint32_t lda = 0, lkc = 0, lch = 0;
    while ((1u << lda) < Da) lda++;
    const size_t S = 2 * N / Da, T = C / (Da * N);
    // a chunk's Da x Da/2 x KC values fill the LDS, or KC is all of S
    while ((Da * Da / 2 << (lkc + 1)) <= 32768 && ((size_t)2 << lkc) <= S) lkc++;
    while (((size_t)1 << (lkc + lch)) < S) lch++;
    if ((Da & (Da - 1)) || Da > 256 || R * T % 8 || (R * T << lch) > 0x7fffffffu) return hipErrorInvalidValue;
    uint32_t Dinv = 0;  // Da^-1 mod 65535 (Da a power of two, odd modulus)
    for (uint32_t x = 1; x < PMOD; x++)
        if ((uint64_t)x * Da % PMOD == 1) { Dinv = x; break; }
    hipLaunchKernelGGL(k_encode, dim3((unsigned)(R * T << lch)), dim3(1024), 0, s, db, (uint32_t)C, (uint32_t)T, lda,
                       lkc, lch, Dinv);
    return hipGetLastError();
}

hipError_t launch_aside(const uint8_t* db, size_t R, size_t C, size_t g0, size_t ng, const uint32_t* crs,
                        uint32_t* a32T, const NttConst& nc, hipStream_t s) {
    hipLaunchKernelGGL(k_aside, dim3((unsigned)(ng * (N / 4))), dim3(512), 0, s, db, (uint32_t)C,
                       (uint32_t)(R / N), (uint32_t)g0, crs, a32T, nc);
    return hipGetLastError();
}

hipError_t launch_ring_embed(uint32_t* a32T, size_t ng, const NttConst& nc, hipStream_t s) {
    hipLaunchKernelGGL(k_ntt_rows, dim3((unsigned)(ng * 2 * N)), dim3(256), 0, s, a32T, nc);
    return hipGetLastError();
}

hipError_t launch_collapse_chain(const uint32_t* F, size_t ng, const uint32_t* ksk5a, uint32_t* dtmp,
                                 uint32_t* states, const NttConst& nc, const CrtConst& cc, hipStream_t s) {
    hipLaunchKernelGGL(k_apost_gather, dim3((unsigned)(ng * 2 * (N / 16))), dim3(1024), 0, s, F, dtmp);
    hipLaunchKernelGGL(k_collapse_chain, dim3((unsigned)ng, 2), dim3(512), 0, s, F, ksk5a, dtmp, states, nc,
                       nr_gadget_const(nc, cc));
    return hipGetLastError();
}

hipError_t launch_collapse_final(const uint32_t* states, size_t ng, const uint32_t* kneg1a, uint32_t* precomp_g0,
                                 const NttConst& nc, const CrtConst& cc, hipStream_t s) {
    hipLaunchKernelGGL(k_collapse_final, dim3((unsigned)ng), dim3(1024), 0, s, states, kneg1a, precomp_g0, nc, cc);
    return hipGetLastError();
}

}  // namespace ipx
