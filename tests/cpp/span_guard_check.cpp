// Host check of the decode's block-span guard (dec_block_span_ok in
// pj_kernels.h): line blocks whose lines span 4 GiB - 1 MiB or more are
// refused, shorter ones pass, whatever the block's position and size.
#include <cstdio>
#include <vector>

#include "pj_kernels.h"

static int fails = 0;
static void expect(bool got, bool want, const char *what) {
    if (got != want) { std::printf("FAIL: %s\n", what); fails++; }
}

// for blocks of lpb lines
static void check(uint64_t lpb) {
    const uint64_t G = 1ull << 30, big = 300 / lpb;
    // 300 lines of 100 bytes, then one line of 4 GiB, then 50 short lines
    std::vector<uint64_t> ls;
    uint64_t a = 0;
    for (int k = 0; k < 300; k++) { ls.push_back(a); a += 100; }
    ls.push_back(a); a += 4 * G;
    for (int k = 0; k < 50; k++) { ls.push_back(a); a += 100; }
    ls.push_back(a);
    const uint64_t lines = ls.size() - 1;
    for (uint64_t b = 0; b * lpb < lines + lpb; b++)
        expect(dec_block_span_ok(ls.data(), lines, lpb, b), b != big, "only the block holding the 4 GiB line spans too much");
    // a block of many lines just under / at the limit
    std::vector<uint64_t> m;
    const uint64_t per = (PJ_DEC_MAX_BLOCK_SPAN - 1) / lpb;
    for (uint64_t k = 0; k <= lpb; k++) m.push_back(k * per);
    expect(dec_block_span_ok(m.data(), lpb, lpb, 0), true, "just under the limit");
    m[lpb] = PJ_DEC_MAX_BLOCK_SPAN;
    expect(dec_block_span_ok(m.data(), lpb, lpb, 0), false, "at the limit");
}

int main() {
    check(104);
    check(64);
    // lines 64 to 127 of 65 MiB: no block of 104 spans too much, one of 64 does
    std::vector<uint64_t> x(1, 0);
    for (int k = 0; k < 300; k++) x.push_back(x.back() + (k >= 64 && k < 128 ? 65ull << 20 : 100));
    for (uint64_t b = 0; b < 3; b++) expect(dec_block_span_ok(x.data(), 300, 104, b), true, "blocks of 104");
    for (uint64_t b = 0; b < 5; b++) expect(dec_block_span_ok(x.data(), 300, 64, b), b != 1, "blocks of 64");
    if (fails) return 1;
    std::printf("span guard checks passed\n");
    return 0;
}
