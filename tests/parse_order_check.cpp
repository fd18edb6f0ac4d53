// parse_order_check.cpp -- the order of the parallel parse's tiles (parse_chunk):
// every row of T workgroups holds one tile of each chunk, and the tiles of each
// chunk (the last one's reach past its stream where the buffer does) fall evenly
// on the eight XCDs, to which the hardware hands workgroups in turn.  Built and
// run by tests/test_parse_order.py with g++; prints "ok <cases>" or the first
// violation.
#include <cstdio>
#include <cstdlib>
#include <vector>

#include "zccl_internal.h"

using namespace zk;

int main()
{
    long cases = 0;
    const uint32_t rows = 512;
    for (uint32_t T = 1; T <= 200; T++) {
        std::vector<uint32_t> on(T * 8, 0);
        for (uint32_t row = 0; row < rows; row++) {
            std::vector<char> seen(T, 0);
            for (uint32_t i = 0; i < T; i++) {
                const uint32_t c = parse_chunk(row, i, T);
                if (c >= T || seen[c]) {
                    std::printf("FAIL T %u row %u: chunk %u twice or out of range\n", T, row, c);
                    return 1;
                }
                seen[c] = 1;
                on[c * 8 + (row * T + i) % 8]++;
            }
        }
        for (uint32_t c = 0; c < T; c++)
            for (uint32_t x = 0; x < 8; x++)
                if (on[c * 8 + x] > rows / 8 * 3 / 2) {
                    std::printf("FAIL T %u: %u of %u tiles of chunk %u on XCD %u\n", T, on[c * 8 + x], rows, c, x);
                    return 1;
                }
        cases++;
    }
    std::printf("ok %ld\n", cases);
    return 0;
}
