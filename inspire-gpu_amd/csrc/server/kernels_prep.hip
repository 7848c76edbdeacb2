// What an answer needs before its passes, in one launch: the flat wire
// query's keys in NTT form with their int8 digits and sums, its RGSW rows,
// and the database pass's operand (int8 digits and sums, or doubles for the
// fp64 pass); every residue reduced mod its limb's prime (the reference
// narrows ksk/RGSW words without reduction, src/gpu_protocol.cu:1066 and :50;
// canonical inputs agree). It also zeroes what later kernels of the answer
// count or add into.
//
// Small tables are bound by launches: as six kernels (unmarshal, key NTT,
// query digits and sums, key digits and sums) this took 24 us of device time
// and 55 us of launches for one query, and 43 us of device time for 32
// (every one of them passing residues through memory).
// One grid of 256-lane workgroups, (role, query): 8 key polynomials, the
// row ranges of the LWE part, 8 eighths of the RGSW part, zeroing. The key
// polynomials, the longest dependent chain, come first. Wire words are read
// once, 8 bytes per lane and coalesced (a caller's buffer need not be
// 16-byte aligned), 16 loads per lane and limb in flight together.
// 32768 rows: one query 5.1 us, 32 queries 14.7 (29 MB read, 12 MB written;
// 17.3 with the digits cut one by one, the limbs' loads one after the other
// and the exchange words zeroed by blocks of their own).
#include "kernels.h"
#include "ntt_regs.h"

namespace ipx {

namespace {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

constexpr size_t BLK = (size_t)D_EFF * 2 * N;
constexpr uint32_t kKeyBlocks = 8;       // (key, digit, limb) polynomials
constexpr uint32_t kRgswWords = 4 * 2 * D_EFF * N;
constexpr uint32_t kRgswBlocks = kRgswWords / 4096;
constexpr uint32_t kChunkRows = 4096;    // LWE rows staged at a time: 16 per lane

// LDS word of staged row r: 4 pad words per 16 put a wave's 16-byte reads
// (16 consecutive rows per lane) on distinct banks
constexpr uint32_t kRowLds = kChunkRows / 16 * 20;
__device__ __forceinline__ uint32_t rl(uint32_t r) { return r + 4 * (r >> 4); }

constexpr uint32_t inv_mod_prime(uint64_t b, uint32_t m) {
    uint64_t r = 1;
    b %= m;
    for (uint64_t e = m - 2; e; e >>= 1, b = b * b % m)
        if (e & 1) r = r * b % m;
    return (uint32_t)r;
}
constexpr uint32_t kQ1InvQ0 = inv_mod_prime(Q1, Q0);

// Balanced base-256 digits of v: adding 128 to every digit but the top one
// makes them plain bytes, and taking it off again flips their top bits. Four
// digits of v < 2^27 (three in [-128, 127], the top in [0, 8]):
__device__ __forceinline__ uint32_t digits4(uint32_t v) { return (v + 0x808080u) ^ 0x808080u; }
// o[k] = byte k of x[0..3]
__device__ __forceinline__ void transpose4(uint32_t (&o)[4], const uint32_t (&x)[4]) {
    const uint32_t a = __builtin_amdgcn_perm(x[1], x[0], 0x05010400u), b = __builtin_amdgcn_perm(x[3], x[2], 0x05010400u);
    const uint32_t c = __builtin_amdgcn_perm(x[1], x[0], 0x07030602u), d = __builtin_amdgcn_perm(x[3], x[2], 0x07030602u);
    o[0] = __builtin_amdgcn_perm(b, a, 0x05040100u);
    o[1] = __builtin_amdgcn_perm(b, a, 0x07060302u);
    o[2] = __builtin_amdgcn_perm(d, c, 0x05040100u);
    o[3] = __builtin_amdgcn_perm(d, c, 0x07060302u);
}

// W: the words of the query, u64 as on the wire or narrowed to u32.
template <typename W>
__global__ __launch_bounds__(256) void k_prep(PrepArgs a, NttConst nc) {
    __shared__ __align__(16) uint32_t lds[2 * kRowLds];  // two limbs of a chunk's rows, or one polynomial
    __shared__ uint64_t red[2][4];
    const uint32_t t = threadIdx.x, qi = blockIdx.y + a.first;
    const W* w = static_cast<const W*>(a.q) + (size_t)qi * a.q_stride;
    const size_t R = a.R;
    uint32_t b = blockIdx.x;
    if (b == 0 && qi == 0) {  // with the first query
        for (uint32_t x = t; x < a.zero_words; x += 256) a.zero[x] = 0;
        if (a.status && t == 0) *a.status = 0;
        if (a.gave_up && t == 0) *a.gave_up = 0;
    }
    if (b < a.key_blocks) {
        // key polynomial b = key*4 + digit*2 + limb
        const int c = (int)(b & 1);
        const uint32_t j = (b >> 1) & 1, key = b >> 2;
        const NrLimb m = nr_limb(c);
        W in[8];
#pragma unroll
        for (int k = 0; k < 8; k++) in[k] = w[a.keys_at + (size_t)b * N + t + 256 * k];
        // the pair chains' exchange words, an eighth per block while the keys load
        u32x4* xz = reinterpret_cast<u32x4*>(a.xbuf + (size_t)qi * a.xbuf_words + b * (a.xbuf_words / kKeyBlocks));
        for (uint32_t x = t; x < a.xbuf_words / kKeyBlocks / 4; x += 256) xz[x] = u32x4{0, 0, 0, 0};
        NrTw tw[4];
        nr_tw_global(tw, nc, c, t);
        uint32_t x[1][8];
#pragma unroll
        for (int k = 0; k < 8; k++) x[0][k] = red64(in[k], c);
        nr_forward1(x, reinterpret_cast<uint32_t(*)[POLY4_LDS]>(lds), tw, t, m);
        uint64_t sum = 0;
#pragma unroll
        for (int k = 0; k < 8; k++) {
            x[0][k] = fold(nr_reduce(x[0][k], m), m.q);
            sum += x[0][k];
        }
        u32x4* o = reinterpret_cast<u32x4*>(a.keys + (size_t)qi * a.keys_stride + (size_t)b * N + 8 * t);
        o[0] = u32x4{x[0][0], x[0][1], x[0][2], x[0][3]};
        o[1] = u32x4{x[0][4], x[0][5], x[0][6], x[0][7]};
        if (key == 0) {
            // kdig[limb][kb][kMp][16 bytes], row m = q*4 + digit of K5 at
            // k = j*N + slot = 16*kb + byte; a lane has 8 bytes of each row.
            // Rows of absent queries keep old bytes: they only reach output
            // rows nobody stores.
            uint32_t d8[2][4], lo[4], hi[4];
#pragma unroll
            for (int e = 0; e < 8; e++) d8[e >> 2][e & 3] = digits4(x[0][e]);
            transpose4(lo, d8[0]);
            transpose4(hi, d8[1]);
            const size_t kb = (size_t)j * (N / 16) + (t >> 1);
            int8_t* d = a.kdig + (((size_t)c * (DD_K / 16) + kb) * a.kMp + (size_t)qi * 4) * 16 + 8 * (t & 1);
#pragma unroll
            for (int k = 0; k < 4; k++) *reinterpret_cast<u32x2*>(d + 16 * k) = u32x2{lo[k], hi[k]};
            const uint64_t s = block_sum_u64<256>(sum, red[0]);
            if (t == 0) a.KS[((size_t)qi * 2 + c) * kKeySumParts + j] = red64(s, c);
        }
        return;
    }
    b -= a.key_blocks;
    if (b < a.lwe_blocks) {
        // rows of part `part`; per-limb digits take one limb per block, the
        // CRT digits (and the doubles) both
        const bool both = a.form != kPrepDigits4;
        const uint32_t part = both ? b : b >> 1, c0 = both ? 0 : b & 1, nl = both ? 2 : 1;
        const uint32_t nkb = (uint32_t)(R / 16);
        const uint32_t kb0 = (uint32_t)((uint64_t)part * nkb / a.parts);
        const uint32_t kb1 = (uint32_t)((uint64_t)(part + 1) * nkb / a.parts);
        uint64_t sum[2] = {0, 0};
        for (uint32_t kc = kb0; kc < kb1; kc += kChunkRows / 16) {
            const uint32_t kn = kb1 - kc < kChunkRows / 16 ? kb1 - kc : kChunkRows / 16, rows = kn * 16;
            if (kc != kb0) __syncthreads();  // the last chunk's rows are read
            // both limbs' words in flight together
            W v[2][16];
#pragma unroll
            for (uint32_t l = 0; l < 2; l++) {
                if (l >= nl) break;
                const W* src = w + (size_t)(c0 + l) * R + (size_t)kc * 16;
#pragma unroll
                for (int i = 0; i < 16; i++) {
                    const uint32_t r = t + 256 * i;
                    v[l][i] = src[r < rows ? r : rows - 1];
                }
            }
#pragma unroll
            for (uint32_t l = 0; l < 2; l++) {
                if (l >= nl) break;
                const int c = (int)(c0 + l);
#pragma unroll
                for (int i = 0; i < 16; i++) {
                    const uint32_t r = t + 256 * i, x = red64(v[l][i], c);
                    if (r < rows) {
                        if (a.form == kPrepDoubles) {
                            a.bq[((size_t)qi * 2 + c) * R + (size_t)kc * 16 + r] = (double)x;
                        } else {
                            sum[l] += x;
                            lds[l * kRowLds + rl(r)] = x;
                        }
                    }
                }
            }
            if (a.form == kPrepDoubles) continue;
            __syncthreads();
            if (t < kn) {
                const size_t kb = kc + t;
                uint32_t x0[16];
#pragma unroll
                for (int g = 0; g < 4; g++) {
                    const u32x4 y = *reinterpret_cast<const u32x4*>(&lds[20 * t + 4 * g]);
#pragma unroll
                    for (int e = 0; e < 4; e++) x0[4 * g + e] = y[e];
                }
                if (a.form == kPrepDigits4) {
                    // dig[kb][Mp][16 bytes], rows m = (2q + limb)*4 + digit
                    u32x4 o[4];
#pragma unroll
                    for (int g = 0; g < 4; g++) {
                        uint32_t d[4], p[4];
#pragma unroll
                        for (int e = 0; e < 4; e++) d[e] = digits4(x0[4 * g + e]);
                        transpose4(p, d);
#pragma unroll
                        for (int k = 0; k < 4; k++) o[k][g] = p[k];
                    }
                    u32x4* d = reinterpret_cast<u32x4*>(a.dig + (kb * a.Mp + ((size_t)2 * qi + c0) * 4) * 16);
#pragma unroll
                    for (int k = 0; k < 4; k++) d[k] = o[k];
                } else {
                    // 7 rows per query: the digits of B = CRT(b_0, b_1) in
                    // [0, Q0*Q1) (six balanced, the top in [0, 32]), row
                    // 7q + digit, or (Mp/7)*digit + q for the power rows
                    u32x4 o[7];
#pragma unroll
                    for (int g = 0; g < 4; g++) {
                        const u32x4 y = *reinterpret_cast<const u32x4*>(&lds[kRowLds + 20 * t + 4 * g]);
                        uint32_t lo[4], hi[4], pl[4], ph[4];
#pragma unroll
                        for (int e = 0; e < 4; e++) {
                            const uint32_t r0 = x0[4 * g + e], r1 = y[e];
                            // Garner: B = r1 + Q1 * ((r0 - r1) * Q1^-1 mod Q0)
                            const uint32_t f = mul_mod(sub_mod(r0, fold(r1, Q0), Q0), kQ1InvQ0, 0);
                            const uint64_t v = (uint64_t)Q1 * f + r1 + 0x808080808080ull;  // as digits4
                            lo[e] = (uint32_t)v ^ 0x80808080u;
                            hi[e] = (uint32_t)(v >> 32) ^ 0x8080u;
                        }
                        transpose4(pl, lo);
                        transpose4(ph, hi);
#pragma unroll
                        for (int k = 0; k < 7; k++) o[k][g] = k < 4 ? pl[k & 3] : ph[k & 3];
                    }
                    u32x4* d = reinterpret_cast<u32x4*>(a.dig + kb * a.Mp * 16);
#pragma unroll
                    for (int k = 0; k < 7; k++) d[a.form == kPrepPower ? a.Mp / 7 * k + qi : 7 * qi + k] = o[k];
                }
            }
        }
        if (a.form == kPrepDoubles) return;
#pragma unroll
        for (uint32_t l = 0; l < 2; l++) {
            if (l >= nl) break;
            const uint64_t s = block_sum_u64<256>(sum[l], red[l]);
            uint32_t* S = a.S + ((size_t)2 * qi + c0 + l) * kOffsetSumParts;
            if (t == 0) S[part] = red64(s, (int)(c0 + l));
            if (part == 0 && t >= a.parts && t < kOffsetSumParts) S[t] = 0;
        }
        return;
    }
    b -= a.lwe_blocks;
    if (b < a.rgsw_blocks) {
        const W* src = w + a.keys_at + 2 * BLK + (size_t)b * 4096;
        uint32_t* dst = a.rgsw + (size_t)qi * a.rgsw_stride + (size_t)b * 4096;
        W v[16];
#pragma unroll
        for (int i = 0; i < 16; i++) v[i] = src[t + 256 * i];
#pragma unroll
        for (int i = 0; i < 16; i++) dst[t + 256 * i] = red64(v[i], i >> 3);  // [..][limb][N]: 4096 words = both limbs
        return;
    }
    // collapse sums a split collapse adds into
    b -= a.rgsw_blocks;
    uint32_t* p2 = a.part2 + (size_t)qi * a.part2_stride + (size_t)b * 4096;
#pragma unroll
    for (int i = 0; i < 4; i++) *reinterpret_cast<u32x4*>(p2 + 4 * (t + 256 * i)) = u32x4{0, 0, 0, 0};
}

}  // namespace

hipError_t launch_prep(PrepArgs a, size_t nq, const DbPlan& p, const NttConst& nc, hipStream_t s, size_t first,
                       size_t count) {
    if (count == 0) count = nq;
    if (first + count > nq) return hipErrorInvalidValue;
    a.first = (uint32_t)first;
    if (nq == 0 || nq > kMfmaMaxQueries || nq > kCollapseMaxQueries || !a.q || a.R == 0 || a.R % N)
        return hipErrorInvalidValue;
    a.Mp = (uint32_t)dbplan_mp(p);
    if (p.kind == DbPlan::F64) {
        if (!a.bq) return hipErrorInvalidValue;
        a.form = kPrepDoubles;
    } else {
        if (!a.dig || !a.S || nq > dbplan_max_queries(p)) return hipErrorInvalidValue;
        a.form = !p.crt ? kPrepDigits4 : p.pow ? kPrepPower : kPrepDigits7;
    }
    // LWE row ranges: 4096 rows each, at most as many as the sums have parts
    size_t parts = (a.R + kChunkRows - 1) / kChunkRows;
    if (parts > kOffsetSumParts) parts = kOffsetSumParts;
    a.parts = (uint32_t)parts;
    a.lwe_blocks = a.skip_lwe ? 0 : (uint32_t)(a.form == kPrepDigits4 ? 2 * parts : parts);
    a.key_blocks = a.rgsw_blocks = 0;
    if (a.keys) {
        if (!a.rgsw || !a.kdig || !a.KS) return hipErrorInvalidValue;
        a.kMp = (uint32_t)collapse_mp(nq);
        a.key_blocks = kKeyBlocks;
        a.rgsw_blocks = kRgswBlocks;
    }
    if (a.part2_words % 4096 || (a.part2_words && !a.part2) || (a.zero_words && !a.zero) ||
        a.xbuf_words % (4 * kKeyBlocks) || (a.xbuf_words && (!a.xbuf || !a.keys)))
        return hipErrorInvalidValue;
    const size_t blocks = a.key_blocks + a.lwe_blocks + a.rgsw_blocks + a.part2_words / 4096;
    const dim3 grid((unsigned)blocks, (unsigned)count);
    if (a.narrow)
        hipLaunchKernelGGL(k_prep<uint32_t>, grid, dim3(256), 0, s, a, nc);
    else
        hipLaunchKernelGGL(k_prep<uint64_t>, grid, dim3(256), 0, s, a, nc);
    return hipGetLastError();
}

}  // namespace ipx
