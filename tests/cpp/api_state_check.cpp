// Host check of pj_api.cpp's own decisions: pj_api.cpp is linked with the HIP
// calls and launches below in place of the runtime and the kernels, so no GPU
// is needed and a line of several GiB costs nothing.
//   * decode: the line blocks that the launches get never span
//     PJ_DEC_MAX_BLOCK_SPAN bytes, and what is refused is decided over the
//     larger blocks whichever are used;
//   * encode: the words that a pass starts from zero are zero at its launch,
//     also when the scratch grew in between and its new memory has the old
//     address; large records get a full grid where their count is not known;
//     a call without room for output launches the size alone.
#include <sys/mman.h>

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <vector>

#include <hip/hip_runtime.h>

#include "petjson.h"
#include "pj_kernels.h"

static int fails = 0;
static void expect(bool ok, const char *what, const char *where) {
    if (!ok) { std::printf("FAIL: %s: %s\n", where, what); fails++; }
}

// ------------------------------------------------------------- the runtime
// Device memory: eight slots of address space, the lowest free one each time,
// so that an allocation after a free has the freed address.  New memory
// starts with other bytes than zero.
constexpr size_t SLOT = 4ull << 30;
constexpr int SLOTS = 8;
static uint8_t *arena;
static bool slot_used[SLOTS];

extern "C" {
hipError_t hipMalloc(void **p, size_t n) {
    if (!arena) {
        void *m = mmap(nullptr, SLOT * SLOTS, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0);
        if (m == MAP_FAILED) return hipErrorOutOfMemory;
        arena = static_cast<uint8_t *>(m);
    }
    if (n > SLOT) return hipErrorOutOfMemory;
    for (int k = 0; k < SLOTS; k++)
        if (!slot_used[k]) {
            slot_used[k] = true;
            *p = arena + k * SLOT;
            std::memset(*p, 0xA5, std::min<size_t>(n, 1 << 20));
            return hipSuccess;
        }
    return hipErrorOutOfMemory;
}
hipError_t hipFree(void *p) {
    slot_used[(static_cast<uint8_t *>(p) - arena) / SLOT] = false;
    return hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t n, unsigned) { return (*p = std::calloc(1, n)) ? hipSuccess : hipErrorOutOfMemory; }
hipError_t hipHostFree(void *p) { std::free(p); return hipSuccess; }
hipError_t hipGetDeviceCount(int *n) { *n = 1; return hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600 *p, int) {
    std::memset(p, 0, sizeof *p);
    std::strcpy(p->gcnArchName, "gfx950");
    return hipSuccess;
}
hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t, int) { *v = 100000; return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) { *s = nullptr; return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { *e = nullptr; return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
const char *hipGetErrorString(hipError_t) { return "error"; }
hipError_t hipPointerGetAttributes(hipPointerAttribute_t *, const void *) { return hipErrorInvalidValue; }
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind) { std::memcpy(d, s, n); return hipSuccess; }
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t) { std::memcpy(d, s, n); return hipSuccess; }
}

// ------------------------------------------------------------ the launches
static std::vector<uint64_t> starts;     // of the decode's lines, and the end
static std::vector<int> parsed_blocks;   // lines per block of each validating launch
static const char *where_now = "";

int pj_dec_index_block() { return 2048; }
int pj_dec_parse_block() { return 104; }
int pj_dec_bscan_block() { return 1024; }
int pj_dec_split_block(uint64_t len, uint64_t lines) { return len > 295 * lines ? 64 : 104; }
uint64_t pj_arr_blocks(uint64_t n) { return (n + 255) / 256; }
uint64_t pj_arr_threads(uint64_t n) { return pj_arr_blocks(n) * 256; }
int pj_decode_model_block() { return 128; }
int pj_encode_block_records(bool nested) { return nested ? 96 : 256; }
int pj_encode_model_records() { return 512; }
int pj_encode_pretty_records() { return 256; }
int pj_encode_rows_size_records() { return 512; }
int pj_encode_pretty_tile_records() { return 64; }
uint64_t pj_select_blocks(uint64_t n) { return (n + 4095) / 4096; }
hipError_t pj_noalloc_scratch_init(int, uint64_t **p) { *p = nullptr; return hipSuccess; }

hipError_t pj_launch_fill_u64(uint64_t *p, uint64_t n, uint64_t v, hipStream_t, uint64_t *) {
    for (uint64_t i = 0; i < n; i++) p[i] = v;
    return hipSuccess;
}
hipError_t pj_launch_fill_ranges(const FillRanges &R, hipStream_t st, uint64_t *) {
    for (int k = 0; k < R.k; k++) (void)pj_launch_fill_u64(R.p[k], R.n[k], R.v[k], st, nullptr);
    return hipSuccess;
}
hipError_t pj_launch_publish(uint64_t *host, uint64_t *src, int n, uint64_t zero, int keep, hipStream_t, uint64_t *) {
    for (int i = 0; i < n; i++) host[i] = src[i];
    for (uint64_t i = 0; i < zero; i++)
        if ((int64_t)i != keep) src[i] = 0;
    return hipSuccess;
}
hipError_t pj_launch_dec_index(const DecParams &P, hipStream_t) {
    for (size_t k = 0; k < starts.size() && k < P.ls_cap; k++) P.line_start[k] = starts[k];
    *P.n_lines = starts.size() - 1;
    return hipSuccess;
}
hipError_t pj_launch_dec_span_check(const DecParams &P, uint64_t *flag, hipStream_t) {
    const uint64_t lpb = P.lpb ? (uint64_t)P.lpb : (uint64_t)pj_dec_parse_block();
    for (uint64_t b = 0; b * lpb < P.lines; b++)
        if (!dec_block_span_ok(P.line_start, P.lines, lpb, b)) *flag = 1;
    return hipSuccess;
}
hipError_t pj_launch_dec_parse(const DecParams &P, hipStream_t) {
    parsed_blocks.push_back(P.lpb);
    expect(P.nblocks == (P.lines + P.lpb - 1) / P.lpb, "block count", where_now);
    for (uint64_t b = 0; b < P.nblocks; b++)
        if (!dec_block_span_ok(P.line_start, P.lines, (uint64_t)P.lpb, b)) {
            expect(false, "a line block at the launch spans too much", where_now);
            break;
        }
    return hipSuccess;
}
hipError_t pj_launch_dec_bscan(const DecParams &, hipStream_t) { return hipSuccess; }
hipError_t pj_launch_dec_write(const DecParams &, hipStream_t) { return hipSuccess; }
hipError_t pj_launch_dec_long(const DecParams &, hipStream_t) { return hipSuccess; }
hipError_t pj_launch_dec_errcode(const DecParams &, hipStream_t) { return hipSuccess; }

static uint64_t large_records;           // that the pass lists
// The pass: its ticket, counters and look-back words must be zero; it leaves
// them as a pass does.
hipError_t pj_launch_encode(const EncParams &P, bool nested, bool, hipStream_t) {
    uint64_t *sc = reinterpret_cast<uint64_t *>(P.ticket);
    const uint64_t nblk = (P.n + pj_encode_block_records(nested) - 1) / pj_encode_block_records(nested);
    for (uint64_t i = 0; i < nblk + 4 && !P.geo; i++)
        if (sc[i]) {
            expect(false, "a word that the pass starts from zero is not zero", where_now);
            break;
        }
    sc[0] = P.order_by_id ? 0 : nblk;
    *P.total = 100;
    if (P.big_cap) *P.big_count = large_records;
    for (uint64_t i = 0; i < nblk; i++) P.state[i] = (2ull << 62) | 100;
    return hipSuccess;
}
static std::vector<bool> big_grids;      // full or not, of each launch for the large records
hipError_t pj_launch_encode_big(const EncParams &, bool full, hipStream_t) {
    big_grids.push_back(full);
    return hipSuccess;
}
static int size_launches;
hipError_t pj_launch_rows_size(const EncParams &P, bool, hipStream_t) {
    size_launches++;
    *P.total = 100;
    return hipSuccess;
}
hipError_t pj_launch_select_status(const EncParams &P, uint32_t, uint64_t *, hipStream_t) {
    *P.total = P.c.n_pets;
    return hipSuccess;
}
hipError_t pj_launch_encode_measure(const EncParams &P, hipStream_t) { *P.ticket = 1; return hipSuccess; }
#define UNUSED_LAUNCH(name, ...) \
    hipError_t name(__VA_ARGS__) { expect(false, #name " launched", where_now); return hipSuccess; }
UNUSED_LAUNCH(pj_launch_add_u64, uint64_t *, uint64_t, uint64_t, hipStream_t)
UNUSED_LAUNCH(pj_launch_put_bytes, uint8_t *, uint32_t, int, hipStream_t)
UNUSED_LAUNCH(pj_launch_copy_pieces, const CopyPieces &, hipStream_t)
UNUSED_LAUNCH(pj_launch_arr_frame, const DecParams &, hipStream_t)
UNUSED_LAUNCH(pj_launch_encode_rows, const EncParams &, bool, hipStream_t)
UNUSED_LAUNCH(pj_launch_encode_pretty, const EncParams &, hipStream_t)
UNUSED_LAUNCH(pj_launch_encode_model, const ModelEncParams &, hipStream_t)
UNUSED_LAUNCH(pj_launch_decode_model, const ModelDecParams &, int, hipStream_t)

// ------------------------------------------------------------------ checks
static uint64_t dev[64];                 // stands for every column: never read

struct Lines {
    std::vector<uint64_t> n;             // line lengths
    Lines &add(uint64_t count, uint64_t bytes) { n.insert(n.end(), count, bytes); return *this; }
};

// Decodes lines of these lengths; blocks is what the launch must get (0: the
// call must be refused).
static void decode(pj_ctx *ctx, const char *what, const Lines &L, int blocks) {
    where_now = what;
    starts.assign(1, 0);
    for (uint64_t b : L.n) starts.push_back(starts.back() + b);
    parsed_blocks.clear();
    pj_pet_columns o;
    std::memset(&o, 0, sizeof o);
    void **v = reinterpret_cast<void **>(&o.id);
    for (int k = 0; k < 17; k++) v[k] = dev;
    pj_decode_result r;
    const pj_status s = pj_decode_device(ctx, reinterpret_cast<uint8_t *>(dev), starts.back(), &o, nullptr, nullptr, 0, &r);
    if (blocks) {
        expect(s == PJ_OK, "accepted", what);
        expect(parsed_blocks.size() == 1 && parsed_blocks[0] == blocks, "lines per block", what);
    } else {
        expect(s == PJ_ERR_INVALID_ARG, "refused", what);
        expect(parsed_blocks.empty(), "nothing launched", what);
    }
}

static void span_guard(pj_ctx *ctx) {
    const uint64_t M = 1ull << 20, G = 1ull << 30;
    for (int tape = 1; tape >= 0; tape--) {
        setenv("PETJSON_DECODE_TAPE", tape ? "1" : "0", 1);
        const int small = tape ? 64 : 104;
        decode(ctx, "short lines, below the limit", Lines().add(1000, 200), 104);
        decode(ctx, "long lines, below the limit", Lines().add(1000, 400), small);
        decode(ctx, "20 MiB lines", Lines().add(300, 20 * M), small);
        // blocks of 64 lines that no block of 104 holds whole
        decode(ctx, "lines 64 to 127 of 65 MiB", Lines().add(64, 100).add(64, 65 * M).add(500, 100), 104);
        decode(ctx, "lines 103 and 104 of 2.2 GiB", Lines().add(103, 100).add(2, 2 * G + 200 * M).add(103, 100), 104);
        decode(ctx, "3 GiB on both sides of line 104", Lines().add(64, 100).add(40, 75 * M).add(24, 125 * M).add(80, 100), 104);
        // refused over 104 lines, though 64 would hold them
        decode(ctx, "60 MiB lines", Lines().add(208, 60 * M), 0);
        decode(ctx, "a line of 4 GiB", Lines().add(300, 100).add(1, 4 * G).add(50, 100), 0);
        decode(ctx, "2.2 GiB lines in one block", Lines().add(64, 100).add(2, 2 * G + 200 * M).add(300, 100), 0);
    }
    unsetenv("PETJSON_DECODE_TAPE");
}

static void scratch_zero(pj_ctx *ctx) {
    pj_pet_columns flat;
    std::memset(&flat, 0, sizeof flat);
    flat.id = reinterpret_cast<int64_t *>(dev);
    flat.name_off = dev;
    flat.name_bytes = reinterpret_cast<uint8_t *>(dev);
    pj_pet_columns nested = flat;
    nested.photo_off = dev;
    nested.url_off = dev;
    nested.url_bytes = reinterpret_cast<uint8_t *>(dev);
    auto encode = [&](const char *what, const pj_pet_columns &from, uint64_t n) {
        where_now = what;
        pj_pet_columns c = from;
        c.n_pets = n;
        uint64_t len = 0;
        expect(pj_encode_device(ctx, &c, PJ_FORMAT_ARRAY, reinterpret_cast<uint8_t *>(dev), sizeof dev, &len) == PJ_OK &&
                   len == 100, "encode", what);
    };
    encode("flat", flat, 100000);                     // 391 blocks, the words cleared behind it
    encode("flat again", flat, 90000);
    encode("nested, the scratch grows for the large-record list", nested, 30000);
    encode("nested again", nested, 20000);
    encode("flat, past what is cleared ahead", flat, 2000000);
    encode("flat, small", flat, 20);
    encode("nested, grows again", nested, 900000);
    encode("nested, small", nested, 20);
}

// Large records that the pass lists are written behind it.  Where its count
// is not waited for, their launch has a full grid unless the last nested
// encode is known to have listed none.
static void large_record_launches() {
    pj_status st;
    pj_ctx *ctx = pj_create(0, &st);
    pj_pet_columns c;
    std::memset(&c, 0, sizeof c);
    c.n_pets = 1000;
    c.id = reinterpret_cast<int64_t *>(dev);
    c.name_off = c.photo_off = c.url_off = dev;
    c.name_bytes = c.url_bytes = reinterpret_cast<uint8_t *>(dev);
    auto encode = [&](const char *what, uint64_t large, bool two_pass, std::vector<bool> want) {
        where_now = what;
        large_records = large;
        big_grids.clear();
        if (two_pass) setenv("PETJSON_ENC_TWO_PASS", "1", 1);
        uint64_t len = 0;
        expect(pj_encode_device(ctx, &c, PJ_FORMAT_ARRAY, reinterpret_cast<uint8_t *>(dev), sizeof dev, &len) == PJ_OK,
               "encode", what);
        unsetenv("PETJSON_ENC_TWO_PASS");
        expect(big_grids == want, "launches for large records", what);
    };
    encode("two passes, the context's first call", 9, true, {true});
    pj_destroy(ctx);
    ctx = pj_create(0, &st);
    encode("one pass, none listed", 0, false, {});
    encode("two passes after none", 0, true, {false});
    encode("one pass, the first large records", 9, false, {true});
    encode("one pass after some", 0, false, {true});
    encode("two passes after some", 9, true, {true});
    for (int k = 0; k < 15; k++) encode("recent", 0, false, {true});
    encode("no longer recent", 0, false, {true});
    encode("none for long", 0, false, {});
    large_records = 0;
    pj_destroy(ctx);
}

// Selections and flat pretty records: a call without room for output launches
// the size alone (the writer is an UNUSED_LAUNCH).
static void size_without_room(pj_ctx *ctx) {
    pj_pet_columns c;
    std::memset(&c, 0, sizeof c);
    c.id = reinterpret_cast<int64_t *>(dev);
    c.name_off = dev;
    c.name_bytes = reinterpret_cast<uint8_t *>(dev);
    c.n_pets = 1000;
    uint64_t len = 0, m = 0;
    for (int format : {PJ_FORMAT_ARRAY, PJ_FORMAT_NDJSON, PJ_FORMAT_PRETTY}) {
        where_now = "selection, no room";
        size_launches = 0;
        expect(pj_encode_by_status_device(ctx, &c, 1, format, nullptr, 0, &len, &m) == PJ_ERR_CAPACITY && len == 100 &&
                   m == 1000 && size_launches == 1, "the size alone", where_now);
    }
    where_now = "flat pretty, no room";
    size_launches = 0;
    expect(pj_encode_device(ctx, &c, PJ_FORMAT_PRETTY, nullptr, 0, &len) == PJ_ERR_CAPACITY && len == 100 &&
               size_launches == 1, "the size alone", where_now);
}

int main() {
    large_record_launches();
    pj_status s;
    pj_ctx *ctx = pj_create(0, &s);
    if (!ctx) { std::printf("FAIL: no context\n"); return 1; }
    scratch_zero(ctx);
    span_guard(ctx);
    size_without_room(ctx);
    pj_destroy(ctx);
    if (fails) return 1;
    std::printf("api state checks passed\n");
    return 0;
}
