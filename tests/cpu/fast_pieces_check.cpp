// The launches of a fast batch's block list (fast_piece), as the launch loop walks them: they cover every
// block once, in order, each launch holds fewer than 2^32 threads, and the kernel's order of a launch's
// blocks reaches each of its blocks exactly once.
#include <cstdio>
#include <vector>

#include "../../include/birp.h"
#include "../../birp_cpp_amd/csrc/birp_internal.h"

using namespace birp;

static int block_of(int b) {  // k_render_fast's place of launch block b
    const int chunk = BIRP_FAST_CHUNK, turn = b >> 3;
    return (turn / chunk * 8 + (b & 7)) * chunk + turn % chunk;
}

int main() {
    const int totals[] = {1, 127, 128, 129, BIRP_FAST_PIECE - 1, BIRP_FAST_PIECE, BIRP_FAST_PIECE + 1, (1 << 24) - 1, 1 << 24, (1 << 24) + 5, INT32_MAX};
    for (int total : totals) {
        long long next = 0;
        for (int first = 0; first < total;) {
            const FastPiece p = fast_piece(total, first);
            if (p.first != next || p.count < 1 || (long long)p.first + p.count > total) return printf("total %d: piece %d + %d after %lld\n", total, p.first, p.count, next), 1;
            if ((unsigned long long)p.grid * 256 >= 1ull << 32 || p.grid < (unsigned)p.count || p.grid % (8 * BIRP_FAST_CHUNK))
                return printf("total %d: grid %u for %d blocks\n", total, p.grid, p.count), 1;
            next += p.count;
            if (total <= BIRP_FAST_PIECE + 1) {
                std::vector<char> seen(p.count, 0);
                for (unsigned b = 0; b < p.grid; b++) {
                    const int at = block_of((int)b);
                    if (at >= p.count) continue;
                    if (seen[at]++) return printf("total %d: block %d twice\n", total, at), 1;
                }
                for (int at = 0; at < p.count; at++)
                    if (!seen[at]) return printf("total %d: block %d never\n", total, at), 1;
            }
            if (total - first <= p.count) break;
            first += p.count;
        }
        if (next != total) return printf("total %d: %lld blocks covered\n", total, next), 1;
    }
    puts("ok");
    return 0;
}
