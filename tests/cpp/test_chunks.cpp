// Checks layout_chunks (inspire-gpu_amd/csrc/server/chunks.h) on the CPU:
// chunks cover every group once, each chain's groups run from the highest to
// the lowest, and every launch of one chain is on one stream.
#include <cstdio>
#include <cstdlib>
#include <vector>

#include "chunks.h"

using inspire::ChunkLayout;

static size_t checked = 0;

static void check(size_t G, size_t D, size_t gchunk, bool head, bool tail) {
    const size_t Da = D < G ? D : G, T = (G + Da - 1) / Da;
    const ChunkLayout l = inspire::layout_chunks(G, T, Da, gchunk, head, tail);
    std::vector<int> stream(T, -1);
    std::vector<size_t> next(T);  // one past the group the chain takes next
    for (size_t t = 0; t < T; t++) next[t] = (t + 1) * Da < G ? (t + 1) * Da : G;
    size_t groups = 0;
    for (size_t k = 0; k < l.chunks.size(); k++) {
        const size_t lo = l.chunks[k].first, hi = l.chunks[k].second;
        const char* what = nullptr;
        if (lo >= hi || hi > G) what = "an empty or overlong chunk";
        for (size_t g = hi; !what && g-- > lo;) {  // as the chains of this chunk's launches take them
            const size_t t = g / Da;
            if (next[t] != g + 1) what = "groups out of order";
            next[t] = g;
            if (stream[t] >= 0 && stream[t] != (int)l.aside(k)) what = "a chain on two streams";
            stream[t] = l.aside(k);
            groups++;
        }
        if (what) {
            std::printf("G %zu D %zu chunk %zu head %d tail %d: %s at [%zu, %zu)\n", G, D, gchunk, head, tail, what,
                        lo, hi);
            std::exit(1);
        }
    }
    if (groups != G) {
        std::printf("G %zu D %zu chunk %zu: %zu groups\n", G, D, gchunk, groups);
        std::exit(1);
    }
    checked++;
}

int main() {
    for (size_t D : {(size_t)256, (size_t)8})
        for (size_t G = 1; G <= (D == 8 ? 80u : 9u * 256); G += G < 64 ? 1 : D == 8 ? 8 : 64)
            for (size_t c = 1; c <= G; c++)
                if (G % c == 0)
                    for (int sp = 0; sp < 4; sp++) check(G, D, c, sp & 1, sp & 2);
    std::printf("%zu layouts checked\n", checked);
    return 0;
}
