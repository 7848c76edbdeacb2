// Wire residues (u64 words) narrowed to the 32-bit words the server stages.
#pragma once
#include <cstddef>
#include <cstdint>

namespace inspire {

// d[i] = s[i] where s[i] < 2^32, else s[i] mod q (the server reduces every
// residue mod q, so both stand for the same one).
void narrow_residues(const uint64_t* s, uint32_t* d, size_t n, uint64_t q);

}  // namespace inspire
