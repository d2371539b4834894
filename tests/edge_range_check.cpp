// Host check of edge_range.h against 64-bit arithmetic; prints "ok" or the first difference.
#include <cstdint>
#include <cstdio>
#include <initializer_list>

#include "edge_range.h"

using namespace medusa;

static int bad(const char* what, uint64_t a, uint64_t b, uint64_t c) {
    std::printf("%s: %llu %llu %llu\n", what, (unsigned long long)a, (unsigned long long)b, (unsigned long long)c);
    return 1;
}

int main() {
    const uint64_t top = 0xFFFFFFFFull;  // the largest end of an edge array
    const uint64_t ends[] = {0, 1, 3, 64, 255, 256, 257, 1000, top - 300, top - 256, top - 64, top - 1, top};
    const uint64_t lens[] = {0, 1, 2, 3, 4, 5, 63, 64, 65, 255, 256, 257, 1023, 1024, 1025, 5000};
    const uint64_t steps[] = {1, 4, 64, 256, 1024};
    for (uint64_t end : ends)
        for (uint64_t len : lens) {
            if (len > end) continue;
            const uint64_t begin = end - len;
            for (uint64_t off : {0ull, 1ull, 3ull, 63ull, 64ull, 768ull, 1023ull, 5000ull}) {
                if (lies_before((uint32_t)begin, (uint32_t)off, (uint32_t)end) != (begin + off < end))
                    return bad("lies_before", begin, off, end);
                const uint64_t want = begin + off < end ? begin + off : end;
                if (advance_to((uint32_t)begin, (uint32_t)off, (uint32_t)end) != want)
                    return bad("advance_to", begin, off, end);
            }
            // a walk as the kernels make it: every position once, and it ends
            for (uint64_t step : steps) {
                uint64_t seen = 0, rounds = 0;
                for (uint32_t k = (uint32_t)begin; k < (uint32_t)end; k = advance_to(k, (uint32_t)step, (uint32_t)end)) {
                    if (++rounds > len) return bad("walk does not end", begin, step, end);
                    for (uint32_t lane = 0; lane < step; ++lane)
                        if (lies_before(k, lane, (uint32_t)end)) {
                            if ((uint64_t)k + lane != begin + seen) return bad("walk order", begin, step, end);
                            ++seen;
                        }
                }
                if (seen != len) return bad("walk count", begin, step, end);
            }
        }
    for (uint64_t count : {0ull, 1ull, 15ull, 16ull, 17ull, 5000ull, (unsigned long long)top - 4095, (unsigned long long)top})
        for (uint64_t begin : {0ull, 7ull, (unsigned long long)top - count})
            for (uint32_t parts : {1u, 8u, 16u, 1000u, 4096u}) {
                if (begin + count > top) continue;
                uint64_t at = begin;
                for (uint32_t p = 0; p < parts; ++p) {
                    const EdgePart E = edge_part((uint32_t)begin, (uint32_t)count, p, parts);
                    if (E.lo != at || E.hi < E.lo) return bad("edge_part", begin, count, p);
                    at = E.hi;
                }
                if (at != begin + count) return bad("edge_part end", begin, count, parts);
            }
    std::printf("ok\n");
    return 0;
}
