// Walks of csrc/k_chunks.h as the exact score kernel makes them: every element
// of k is in exactly one chunk, around the chunk's length and past 2^31. Built
// and run on the CPU; makes no HIP call.
#include <cstdio>

#include "k_chunks.h"

int main() {
    const int64_t two31 = int64_t(1) << 31;
    for (int64_t k : {int64_t(1), int64_t(31), int64_t(32), int64_t(33), int64_t(64), int64_t(100), two31 - 33, two31 - 1, two31,
                      two31 + 1, two31 + 40, 2 * two31, 2 * two31 + 7}) {
        int64_t elements = 0, chunks = 0;
        for (ofh::KChunks<32> c(k); c.any(); c.next()) {
            if (c.len() <= 0 || c.len() > 32 || c.more() != (elements + c.len() < k)) return std::printf("bad chunk, k %lld\n", (long long)k), 1;
            elements += c.len();
            ++chunks;
        }
        if (elements != k || chunks != (k + 31) / 32) return std::printf("k %lld: %lld elements\n", (long long)k, (long long)elements), 1;
    }
    std::printf("ok\n");
    return 0;
}
