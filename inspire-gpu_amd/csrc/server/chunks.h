// The group chunks of a pipelined answer, and which of the two chain streams
// a chunk's Horner steps run on (host code, no device types).
#pragma once
#include <cstddef>
#include <utility>
#include <vector>

namespace inspire {

struct ChunkLayout {
    // [lo, hi) in launch order, every chain's highest groups first
    std::vector<std::pair<size_t, size_t>> chunks;
    // Every chunk lies in one response ciphertext, so two ciphertexts' chains
    // may advance on two streams. Otherwise a chunk continues one chain and
    // starts the next: a chain's launches then have only their stream to
    // order them, and all of them take the same one.
    bool by_ct = false;
    size_t Da = 0, T = 1;
    // Whether chunk k's chains run on the second stream (where it is free).
    bool aside(size_t k) const { return by_ct && (T - 1 - chunks[k].first / Da) % 2 == 1; }
};

// G groups in T chains of Da (the last may be shorter), gchunk dividing G.
// The chunks of every response ciphertext's chain, highest first, taken in
// turns where chunks end with the ciphertexts: the chains of several then
// advance side by side, and only a chunk's steps of each are left after the
// last pass. The highest chunk splits in 1/4, 1/4, 1/2 with head_split, the
// lowest in 1/2, 1/4, 1/4 with tail_split.
inline ChunkLayout layout_chunks(size_t G, size_t T, size_t Da, size_t gchunk, bool head_split, bool tail_split) {
    ChunkLayout out;
    out.Da = Da;
    out.T = T;
    out.by_ct = T > 1 && G % T == 0 && G / T == Da && Da % gchunk == 0;
    const size_t nct = out.by_ct ? T : 1, per = G / nct, n = per / gchunk, h = gchunk / 2, q = gchunk / 4;
    const bool quarters = G > gchunk && gchunk % 4 == 0;
    std::vector<std::vector<std::pair<size_t, size_t>>> lists(nct);
    for (size_t ct = 0; ct < nct; ct++)
        for (size_t k = n; k-- > 0;) {
            const size_t lo = ct * per + k * gchunk, hi = lo + gchunk;
            auto& l = lists[ct];
            if (quarters && head_split && hi == G) {
                l.push_back({hi - q, hi});
                l.push_back({hi - h, hi - q});
                l.push_back({lo, hi - h});
            } else if (quarters && tail_split && lo == 0) {
                l.push_back({lo + h, hi});
                l.push_back({lo + q, lo + h});
                l.push_back({lo, lo + q});
            } else {
                l.push_back({lo, hi});
            }
        }
    for (size_t r = 0, left = nct; left; r++) {
        left = 0;
        for (size_t ct = nct; ct-- > 0;)
            if (r < lists[ct].size()) {
                out.chunks.push_back(lists[ct][r]);
                left++;
            }
    }
    return out;
}

}  // namespace inspire
