// The host side of the verify path above the kernels: Backend::matvec, the device entry points, and the session's MoE /
// head / acceptance operations.  Mirrors the hot subset of crates/shadowzero-cuda/src/{backend.rs,session.rs}.
#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <cstring>
#include <initializer_list>
#include <map>
#include <string>
#include <unordered_map>
#include <utility>
#include <vector>

#include "sz_internal.hpp"

namespace sz {

// ---- formats ------------------------------------------------------------------------------------------------------
bool format_of(int ty, Format& f, std::string& tag) {
    f = Format{};
    if (ty == SZ_TYPE_Q8_0) {
        f.qk = 32; f.bb = 34; tag = "q8_0";
    } else if (ty == SZ_TYPE_IQ3_S) {
        f.qk = 256; f.bb = 110; tag = "iq3_s";
    } else if (ty == SZ_TYPE_F32 || ty == SZ_TYPE_F16 || ty == SZ_TYPE_BF16) {
        f.dense = true; f.qk = 1; f.bb = ty == SZ_TYPE_F32 ? 4 : 2; tag = ty == SZ_TYPE_F32 ? "f32" : ty == SZ_TYPE_F16 ? "f16" : "bf16";
    } else if (ty >= 1021 && ty <= 1028) {
        f.exl3 = true; f.bits = ty - 1020; tag = "exl3_" + std::to_string(f.bits);
    } else if (ty >= 1031 && ty <= 1033) {
        f.exl3 = true; f.half = true; f.bits = ty - 1030; tag = "exl3h_" + std::to_string(f.bits);
    } else {
        return false;
    }
    f.tag = tag.c_str();
    return true;
}

uint64_t matrix_bytes(const Format& f, uint64_t cols, uint64_t rows) {
    if (f.exl3) return 2 * cols + 2 * rows + 4 + cols * rows * (uint64_t) (2 * f.bits + (f.half ? 1 : 0)) / 16;   // exl3.rs:390-393
    return rows * (cols / f.qk) * f.bb;
}

// Rows a workgroup of the staged GGUF kernels takes: about `lds` bytes of LDS (up to 40 KB for rows of more than 64 units), a
// multiple of 4 * (rows side by side in a wave), at most `cap` where that is such a multiple.
uint32_t rows_per_block(const Format& f, uint32_t cols, uint32_t cap, uint32_t lds) {
    if (f.exl3 || f.dense || cols == 0 || cols % f.qk || cols % 32) return 0;
    const uint32_t units = cols / 32;
    const uint32_t rb = cols / f.qk * f.bb;
    uint32_t ul = 64;                       // lanes a row takes in a wave (rows_body in kernels/matvec.hip)
    if (units < 64)
        for (ul = 1; ul < units;) ul *= 2;
    const uint32_t rg = 64 / ul;
    const uint32_t quantum = 4 * rg;
    uint32_t rpb = (lds / rb) / quantum * quantum;
    if (units > 64) rpb = 8 * rb <= 40960 ? 8 : 4;   // wide rows: 8 where they fit, so that the inputs are staged half as often (measured)
    if (rpb == 0) rpb = quantum;
    if ((uint64_t) rpb * rb + 32 + rpb * 16 > 60000) return 0;
    rpb = std::min<uint32_t>(rpb, units > 64 ? 16 : 64);   // rows_wide keeps the sums of at most 4 rows a wave
    if (rpb > cap) rpb = std::max(quantum, cap / quantum * quantum);
    return rpb;
}

// How the unquantized-matrix kernels split a row of `cols` columns (dense_waves and dense_lanes in kernels/matvec.hip): waves a
// row, threads a workgroup and rows a workgroup takes at a time; the kernels' variant for m inputs; their type code.
struct DenseShape {
    uint32_t waves, block, pass;
};
DenseShape dense_shape(uint64_t cols) {
    uint32_t g = 64;
    while (g > 1 && (uint64_t) (g / 2) * 16 >= cols) g /= 2;
    const uint32_t waves = (uint32_t) std::min<uint64_t>(8, (cols + 1023) / 1024), block = 64 * std::max<uint32_t>(4, waves);
    return {waves, block, block / 64 / waves * (64 / g)};
}
const char* dense_m(uint32_t m) { return m == 1 ? "1" : m <= 4 ? "4" : "8"; }
uint32_t dense_code(int ty) { return ty == SZ_TYPE_F32 ? 0 : ty == SZ_TYPE_F16 ? 1 : 2; }

// Bytes of LDS a compute unit of the MI355X has.
const uint32_t CU_LDS_BYTES = 160 * 1024;

// Workgroups of a kernel that loops over its work (the head): a few per compute unit of the MI355X's 256.
uint32_t persistent_groups() {
    static const uint32_t n = [] {
        const char* e = std::getenv("SHADOWZERO_HEAD_GROUPS");
        const int v = e ? std::atoi(e) : 0;
        return (uint32_t) (v > 0 ? v : 768);
    }();
    return n;
}

// Partial sums an EXL3 product leaves per output: one wave takes 128 inputs of a 128-output block, the four waves of a
// workgroup add theirs up.
uint32_t exl3_ksplit(uint32_t in_f) { return (in_f / 128 + 3) / 4; }

static int check_exl3_shape(uint64_t in_f, uint64_t out_f) {
    if (in_f == 0 || out_f == 0 || in_f % 128 || out_f % 128) return fail("EXL3 projections need in and out to be multiples of 128");
    return 0;
}

// ---- device scratch that grows on demand (backend.rs:42-52) ---------------------------------------------------------
struct DevBuf {
    uint64_t ptr = 0, bytes = 0;
    int need(uint64_t n) {
        if (bytes >= n) return 0;
        if (ptr) sz_free(ptr);
        ptr = 0;
        bytes = 0;
        if (sz_malloc(&ptr, n)) return 1;
        bytes = n;
        return 0;
    }
    ~DevBuf() {
        if (ptr && initialized()) sz_free(ptr);
    }
};

// The variant of a verify launch over `cols` output columns: column tiles a wave and the kernel name's prefix.  `waves8` is the
// number of waves that 8 tiles a wave would give: they do least work for their A rows but leave SIMDs idle where there are few of
// them.  Measured with 2, 4 and 8 tiles throughout, at K = 3 and 1 to 8 rows, over layers of 512 experts of 512 (top-10), 128 of
// 768 (top-8) and 32 of 1536 (top-4), and rounds of 4 and 16 of them: this choice is within 1.5 % of the best (at 8 rows of 4
// layers of 512: 3 %).  E.g. 4 layers alone at 1, 4 and 8 rows of 512 experts: 97, 167 and 289 us with 2, 115, 172 and 274 with 4,
// 162, 204 and 282 with 8, 97, 166 and 272 here; a round of 16 at 8 rows 734, 658, 617, 617 here; of 32 experts of 1536 1418,
// 1214, 1100, 1095 here.  A projection alone for more than four inputs: cols_variant.
static const char* verify_variant(uint64_t cols, uint64_t waves8, uint32_t m, uint32_t* ct) {
    *ct = cols % 512 == 0 && waves8 >= 8192 ? 8 : cols % 256 == 0 && waves8 >= 2048 ? 4 : 2;
    if (m > 4) return *ct == 8 ? "w_" : *ct == 4 ? "t4w_" : "t2w_";
    return *ct == 8 ? "" : *ct == 4 ? "t4_" : "t2_";
}

// ---- one product y_j = W x_j, j < m, on device pointers ---------------------------------------------------------------
// EXL3 workspace: f32 part[m][ks][rows] (callers have always been asked for more: the size they know stays)
static uint64_t align16(uint64_t v) { return (v + 15) & ~15ull; }

static uint64_t cols_scratch_bytes(const Format& f, uint64_t cols, uint64_t rows, uint32_t m) {
    if (!f.exl3) return 0;
    const uint64_t ng = (m + 3) / 4;
    return align16(ng * 8) + align16(ng * 17 * 4) + ng * exl3_ksplit((uint32_t) cols) * 4 * rows * 4;
}

// The GGUF products of kernels/gguf.hip: a wave a 256-column chunk, the same number of chunks a wave as far as they divide, up to
// 16 waves; the dynamic LDS of a workgroup of so many waves for `tiles` row tiles and 4 ng inputs.
static uint32_t gguf_waves(uint64_t cols) {
    const uint32_t chunks = (uint32_t) ((cols + 255) / 256), each = (chunks + 15) / 16;
    return (chunks + each - 1) / each;
}
static uint32_t gguf_lds(uint32_t waves, uint32_t tiles, uint32_t ng) { return waves * (1584 * 4 + tiles * ng * 64 * 4); }

// The column tiles of a projection alone, by its w blocks of 128 columns and 512 inputs.  Up to four inputs as a verify launch's, but above 5 bits
// one tile where its 2 w workgroups do not outnumber the compute units (EXL3_COLS_NARROW_ENTRIES).
// For more than four inputs a launch has w workgroups of two tiles a wave, w / 2 of four or w / 4 of eight, and lasts as long as the compute units
// that have one more than the others: a unit has n2, n4 or n8 of them at most, and twice the tiles cost 1.6 to 1.9 times as much a workgroup.
// They win where that halves the number, and where it only nearly does the higher the rate and the number of inputs the sooner.  us a call by two, four and eight tiles:
//   w            768              1024             1280             1792             2048             2816             3584             4224
//   n2 n4 n8     3 2 1            4 2 1            5 3 2            7 4 2            8 4 2            11 6 3           14 7 4           17 9 5
//   1 bit,  m 5  16.3 18.3 19.3   19.2 18.9 19.8   22.2 23.8 27.9   28.0 29.1 28.8   30.8 29.7 29.5   40.4 40.2 39.1   49.4 46.2 47.9   57.7 56.1 57.7
//   2 bits, m 5  16.4 18.4 21.2   19.8 19.3 21.8   23.3 23.9 28.8   29.0 29.0 29.7   32.2 29.8 30.2   42.2 40.5 39.6   51.7 46.7 48.6   60.4 56.6 57.9
//           m 8  19.4 20.6 22.9   22.9 21.6 23.6   26.9 26.8 31.1   34.3 32.7 32.5   38.8 34.0 33.3   49.7 45.9 43.8   61.0 52.8 53.4   71.3 62.1 62.8
//   4 bits, m 5  17.4 19.1 21.2   21.5 19.9 21.8   25.1 24.4 29.1   32.1 30.9 30.3   35.9 32.1 30.6   46.5 43.1 40.3   57.5 50.6 51.0   66.9 59.8 59.2
//           m 8  19.9 21.0 23.0   24.3 22.0 23.5   28.5 27.3 31.5   36.6 35.2 33.0   40.7 36.3 33.5   53.1 48.7 44.3   66.0 56.1 55.4   77.7 64.4 62.8
//   8 bits, m 8  22.8 22.0 21.3   27.9 22.8 22.0   33.4 31.7 32.5   44.0 39.0 33.7   49.2 40.9 35.5   65.0 56.1 49.9   80.8 67.0 62.0   95.3 77.7 72.6
// Over all rates, the half ones among them, 5 and 8 inputs and 43 values of w from 512 to 6144 the choice is 0.4 % above the best of the three on the
// average and nowhere more than 1.5 % above that of a verify launch, which is 5.7 % above the best.
static const char* cols_variant(const Format& f, uint64_t cols, uint64_t rows, uint32_t m, uint32_t* ct) {
    const uint64_t w = rows / 128 * exl3_ksplit((uint32_t) cols), n2 = (w + 255) / 256, n4 = (w + 511) / 512, n8 = (w + 1023) / 1024;
    if (m > 4 && w > 768) {
        const bool low = f.bits < 3;
        const bool eight = w >= 2816 && (f.bits >= 5 || (m > 6 && !low));
        if (rows % 512 == 0 && (eight || (n4 == 2 * n8 && (n8 > 2 || (n8 == 2 && (m > 6 || !low)))))) { *ct = 8; return "w_"; }
        const uint64_t four = !low ? 1280 : f.bits == 1 && !f.half ? 2048 : 1281;
        if (rows % 256 == 0 && (n2 == 2 * n4 || w >= four)) { *ct = 4; return "t4w_"; }
    }
    if (!f.half && f.bits >= 6 && cols % 256 == 0 && w <= 128) { *ct = 1; return m > 4 ? "t1w_" : "t1_"; }
    return verify_variant(rows, w, m, ct);
}

int matvec_cols_dev(int ty, uint64_t w, uint64_t cols, uint64_t rows, uint64_t x, uint32_t xs, uint64_t y, uint32_t ys, uint32_t m,
                           uint64_t scratch, uint64_t scratch_bytes, uint64_t stream) {
    Format f;
    std::string tag;
    if (!format_of(ty, f, tag)) return fail("no matvec kernel for ggml type " + std::to_string(ty));
    if (m == 0 || m > 8) return fail("matvec_cols takes 1..8 inputs");
    if (xs < cols || ys < rows) return fail("matvec_cols: row strides shorter than the rows");
    if (cols >> 31 || rows >> 31) return fail("matvec_cols: shape too large");
    if (f.exl3) {
        if (check_exl3_shape(cols, rows)) return 1;
        if (xs % 4 || (x & 15)) return fail("matvec_cols: inputs must be 16-byte aligned");
        if (scratch_bytes < cols_scratch_bytes(f, cols, rows, m) || !scratch) return fail("matvec_cols: workspace too small for EXL3");
        const uint32_t zs = exl3_ksplit((uint32_t) cols);
        uint32_t ct;
        const std::string kn = std::string("matvec_grouped_") + cols_variant(f, cols, rows, m, &ct) + tag;
        const sz_arg a0[] = {P(w), P(x), U32(xs), P(scratch), U32((uint32_t) cols), U32((uint32_t) rows), U32(m)};
        if (launch(kn.c_str(), (uint32_t) rows / (64 * ct), zs, 1, 256, 0, stream, a0)) return 1;
        const sz_arg a1[] = {P(scratch), P(w), P(y), U32(ys), U32((uint32_t) cols), U32((uint32_t) rows)};
        return launch("exl3_finish_rows", (uint32_t) rows / 128, m, 1, 64, 0, stream, a1);
    }
    auto each_alone = [&]() -> int {   // a weight at a time, an input at a time
        const std::string kn = "matvec_" + tag;
        for (uint32_t j = 0; j < m; j++) {
            const sz_arg a[] = {P(w), P(x + (uint64_t) j * xs * 4), P(y + (uint64_t) j * ys * 4), U32((uint32_t) rows), U32((uint32_t) cols)};
            if (launch(cols ? kn.c_str() : "matvec_q8_0", ((uint32_t) rows + 3) / 4, 1, 1, 256, 0, stream, a)) return 1;
        }
        return 0;
    };
    if (f.dense && rows == 0) return 0;
    if (cols == 0) return each_alone();   // empty sums, whatever the type: the launches below divide the columns up
    if (f.dense) {
        if (cols % 4 || (x & 15) || xs % 4 || (w & (4 * f.bb - 1))) return fail("matvec_cols: unquantized matrices need columns in fours and aligned rows");
        // several passes a workgroup once there are more than about 1024 of them: the inputs stay in its registers
        const DenseShape d = dense_shape(cols);
        const uint32_t np = (uint32_t) std::min<uint64_t>(16, std::max<uint64_t>(1, rows / (1024ull * d.pass)));
        const std::string kn = std::string("matvec_cols_dense_m") + dense_m(m);
        const sz_arg a[] = {U32(dense_code(ty)), P(w), P(x), U32(xs), P(y), U32(ys), U32((uint32_t) rows), U32((uint32_t) cols), U32(m), U32(np)};
        return launch(kn.c_str(), (uint32_t) ((rows + (uint64_t) d.pass * np - 1) / ((uint64_t) d.pass * np)), 1, 1, d.block, 0, stream, a);
    }
    if (cols % f.qk) return fail("matvec_cols: columns are not whole blocks");
    if ((x & 15) || xs % 4) return each_alone();   // any alignment
    // as many workgroups as the chip holds at a time (16 waves a CU), each with up to four tiles of 16 rows, which share the work
    // on the inputs
    const uint32_t waves = gguf_waves(cols);
    const uint32_t n16 = (uint32_t) ((rows + 15) / 16), slots = 256 * (16 / waves), rounds = (n16 + 4 * slots - 1) / (4 * slots);
    const uint32_t ng = m > 4 ? 2 : 1;
    const std::string kn = std::string("matvec_cols_") + (m > 4 ? "w_" : "") + tag;
    const sz_arg a[] = {P(w), P(x), U32(xs), P(y), U32(ys), U32((uint32_t) rows), U32((uint32_t) cols), U32(m)};
    return launch(kn.c_str(), std::min(n16, rounds * slots), 1, 1, 64 * waves, gguf_lds(waves, 4, ng), stream, a);
}

}   // namespace sz

using namespace sz;

// ---- B1: Backend ----------------------------------------------------------------------------------------------------
// Pinned host memory that the device reads and writes directly (grown on demand, freed with its owner).
struct PinnedBuf {
    void* ptr = nullptr;
    uint64_t bytes = 0;
    int need(uint64_t n) {
        if (bytes >= n) return 0;
        if (ptr) hip().hipHostFree(ptr);
        ptr = nullptr;
        bytes = 0;
        if (hip_check(hip().hipHostMalloc(&ptr, n, 0), "hipHostMalloc")) return 1;
        bytes = n;
        return 0;
    }
    ~PinnedBuf() {
        if (ptr) hip().hipHostFree(ptr);
    }
};

struct sz_backend {
    uint64_t budget = 0, resident_bytes = 0, uploads = 0;
    std::unordered_map<std::string, DevBuf> resident;
    DevBuf w, x, scratch;
    PinnedBuf hx, hy;   // the call's input on its way to the device, and its output, which the kernel writes here itself
};

extern "C" {

sz_backend* sz_backend_new(uint64_t budget) {
    clear_error();
    if (ensure_init()) return nullptr;
    sz_backend* b = new sz_backend();
    b->budget = budget;
    return b;
}
void sz_backend_free(sz_backend* b) { delete b; }
uint64_t sz_backend_resident_bytes(const sz_backend* b) { return b->resident_bytes; }
uint64_t sz_backend_uploads(const sz_backend* b) { return b->uploads; }

int32_t sz_matvec(sz_backend* b, int32_t ty, uint64_t cols, uint64_t rows, const void* bytes, uint64_t nbytes, const char* key, const float* x,
                  float* y) {
    clear_error();
    if (!b) return fail("sz_matvec: null backend");
    Format f;
    std::string tag;
    if (!format_of(ty, f, tag)) return fail("no matvec kernel for ggml type " + std::to_string(ty));   // the reference panics here (backend.rs:60)
    if (!f.exl3 && (cols == 0 || cols % f.qk)) return fail("sz_matvec: columns are not whole blocks");
    if (!f.exl3 && rows == 0) rows = nbytes / (cols / f.qk * f.bb);
    if (f.exl3 && check_exl3_shape(cols, rows)) return 1;
    if (matrix_bytes(f, cols, rows) != nbytes) return fail("sz_matvec: " + std::to_string(nbytes) + " bytes for " + std::to_string(rows) + " x " + std::to_string(cols) + " of " + tag);
    uint64_t wp = 0;
    if (key) {
        auto it = b->resident.find(key);
        if (it != b->resident.end()) {
            if (it->second.bytes < nbytes) return fail(std::string("sz_matvec: resident tensor ") + key + " is smaller than the bytes given");
            wp = it->second.ptr;
        } else if (b->resident_bytes + nbytes <= b->budget) {
            DevBuf& d = b->resident[key];
            if (d.need(nbytes) || sz_upload(d.ptr, bytes, nbytes)) {
                b->resident.erase(key);
                return 1;
            }
            b->resident_bytes += nbytes;
            b->uploads++;
            wp = d.ptr;
        }
    }
    if (!wp) {
        if (b->w.need(nbytes) || sz_upload(b->w.ptr, bytes, nbytes)) return 1;
        b->uploads++;
        wp = b->w.ptr;
    }
    // x goes through pinned memory with an asynchronous copy and y is written into pinned memory by the kernel itself: the call
    // waits once, for the stream, instead of once a blocking copy each way (31 -> 20 us a call for a resident 1024 x 2048 matrix)
    if (b->x.need(cols * 4) || b->hx.need(cols * 4) || b->hy.need(rows * 4)) return 1;
    std::memcpy(b->hx.ptr, x, cols * 4);
    if (hip_check(hip().hipMemcpyHtoDAsync((void*) b->x.ptr, b->hx.ptr, cols * 4, nullptr), "hipMemcpyHtoDAsync")) return 1;
    const uint64_t sb = cols_scratch_bytes(f, cols, rows, 1);
    if (sb && b->scratch.need(sb)) return 1;
    // fewer rows a workgroup where the launch would otherwise have under about 512 workgroups (two a CU)
    const uint32_t rpb = rows_per_block(f, (uint32_t) cols, (uint32_t) std::max<uint64_t>(1, rows / 512));
    if (rpb) {
        const sz_arg a[] = {P(wp), P(b->x.ptr), P((uint64_t) b->hy.ptr), U32((uint32_t) rows), U32((uint32_t) cols), U32(rpb)};
        if (launch(("matvec_one_" + tag).c_str(), ((uint32_t) rows + rpb - 1) / rpb, 1, 1, 256, rpb * (uint32_t) (cols / f.qk * f.bb) + 32, 0, a)) return 1;
    } else if (matvec_cols_dev(ty, wp, cols, rows, b->x.ptr, (uint32_t) cols, (uint64_t) b->hy.ptr, (uint32_t) rows, 1, b->scratch.ptr, b->scratch.bytes, 0)) return 1;
    if (sz_stream_synchronize(0)) return 1;   // synchronous, as the reference's backend: waits for the kernels
    std::memcpy(y, b->hy.ptr, rows * 4);
    return 0;
}

// ---- B4: device entry points ------------------------------------------------------------------------------------------
int32_t sz_dequantize(int32_t ty, uint64_t w, uint64_t out, uint64_t cols, uint64_t rows, uint64_t stream) {
    clear_error();
    Format f;
    std::string tag;
    if (!format_of(ty, f, tag)) return fail("no dequantizer for ggml type " + std::to_string(ty));
    if (f.exl3) {
        if (check_exl3_shape(cols, rows)) return 1;
        const std::string kn = std::string(f.half ? "exl3_decode_h" : "exl3_decode_") + std::to_string(f.bits);
        const sz_arg a[] = {P(w), P(out), U32((uint32_t) cols), U32((uint32_t) rows)};
        return launch(kn.c_str(), (uint32_t) rows / 128, (uint32_t) cols / 16, 1, 64, 0, stream, a);
    }
    if (f.dense) return fail("sz_dequantize: an unquantized matrix has nothing to dequantize");
    if (cols % f.qk) return fail("sz_dequantize: columns are not whole blocks");
    const uint64_t n = cols * rows;
    if (n == 0) return 0;
    const std::string kn = "dequant_" + tag;
    const sz_arg a[] = {P(w), P(out), U64(n)};
    return launch(kn.c_str(), (uint32_t) ((n + 255) / 256), 1, 1, 256, 0, stream, a);
}

int32_t sz_exl3_codebook(uint64_t out, uint64_t stream) {
    clear_error();
    const sz_arg a[] = {P(out), U32(65536)};
    return launch("exl3_codebook", 256, 1, 1, 256, 0, stream, a);
}

uint64_t sz_matvec_cols_scratch(int32_t ty, uint64_t cols, uint64_t rows, uint32_t m) {
    Format f;
    std::string tag;
    if (!format_of(ty, f, tag)) return 0;
    return cols_scratch_bytes(f, cols, rows, m);
}

int32_t sz_matvec_cols(int32_t ty, uint64_t w, uint64_t cols, uint64_t rows, uint64_t x, uint32_t xs, uint64_t y, uint32_t ys, uint32_t m,
                       uint64_t scratch, uint64_t scratch_bytes, uint64_t stream) {
    clear_error();
    return matvec_cols_dev(ty, w, cols, rows, x, xs, y, ys, m, scratch, scratch_bytes, stream);
}

}   // extern "C"

// ---- B2: the session ----------------------------------------------------------------------------------------------------
struct SzLayer {
    int type = 0, shared_type = 0;
    uint64_t experts = 0, stride = 0, shared = 0;
    uint64_t gap = 0; // bytes between an expert's projections (0: the reference's contiguous [gate|up|down])
    DevBuf eaddr;     // u64[3 * ne] then u64[3] for the shared expert
    uint64_t router = 0, gate = 0;   // the router and the shared expert's gate row (set_router; gate 0: none)
    int router_type = 0, gate_type = 0;
    uint32_t vpos = 0;   // an EXL3 layer's place in the session's table of them
    bool set = false;
};

// An EXL3 layer as the verify launches see it (VerifyLayer of kernels/exl3.hip).
struct VerifyLayer {
    uint64_t experts, stride, shared;
    uint32_t part, layer;
};
static_assert(sizeof(VerifyLayer) == 32, "the kernels read this layout");

struct SzGraphKey {
    uint64_t v[10];
    bool operator<(const SzGraphKey& o) const { return std::memcmp(v, o.v, sizeof v) < 0; }
};

// A captured round: its graph, and where its last layer leaves its routing (last_plan, last_fused below).
struct SzRoundGraph {
    uint64_t exec, plan;
    bool fused;
};

struct sz_session {
    sz_session_config cfg{};
    std::vector<SzLayer> layers;
    int head_type = 0;
    uint64_t head_w = 0;
    // batch buffers (session.rs `bb`): the plan, the expert products, the split-k partials, the head's scratch
    DevBuf plan, eg, act, eo, part, dn, head_part, logits, topv, topi, ids;
    DevBuf plans;                 // a plan a layer for the rounds (sz_verify_round)
    uint32_t plan_stride = 0;
    std::vector<VerifyLayer> vtab;   // the EXL3 layers that are set, by type and then in order; its copy on the device
    DevBuf vtab_dev;
    uint32_t vchunk = 1;             // EXL3 layers that `part` and `dn` hold at a time
    DevBuf head_xa, head_inv;   // an EXL3 head's rotated inputs as f16 high and low parts (16 rows of 128 a 128-block), and the tokens' scales
    DevBuf rl, sgl;   // the router's outputs for a batch: f32[max_rows][n_expert], f32[max_rows]
    // the optional 2-bit screen of an EXL3 head (HeadProxy of session.rs:428-441): k_blk = 0 is off
    struct {
        uint32_t k_blk = 0;
        DevBuf w_q2, w_sc, xq, x_sc, x_corr, bmax, seen, sel, logits;
    } hp;
    // The prefill chunk's buffers: parts of one allocation, grown on demand and laid out anew by every chunk.
    struct {
        struct Part {
            uint64_t ptr = 0;
        };
        DevBuf mem;
        Part xq, xd, xh, tidx, w, cnt, offs, list, items, hq, hh, hd, eo, most, arows, ainv, drows, dinv;
        int lay(std::initializer_list<std::pair<Part*, uint64_t>> parts) {
            uint64_t n = 0;
            for (const auto& p : parts) n += (p.second + 255) & ~255ull;
            if (mem.need(n)) return 1;
            n = mem.ptr;
            for (const auto& p : parts) {
                p.first->ptr = n;
                n += (p.second + 255) & ~255ull;
            }
            return 0;
        }
    } pf;
    void* top_host = nullptr;  // pinned host memory the top-64 merge writes to directly (8 rows of 128 words): no copy back
    bool last_fused = false;   // the last layer call left its routing in the fused layout [tidx | w | cnt]
    uint64_t last_plan = 0;    // the plan the last layer call left its routing in
    std::map<SzGraphKey, SzRoundGraph> graphs;
    // plan offsets for the largest batch
    uint32_t GT_max = 0;
    bool use_graph = true;
};

namespace {

struct PlanLayout {
    uint32_t G, nsh, GT, R, a0, r0, w_off, counts_off, tidx_off, bytes;
};

PlanLayout plan_layout(uint32_t m, uint32_t k) {
    PlanLayout p{};
    p.G = m * k;
    p.nsh = (m + 3) / 4;
    p.GT = p.G + p.nsh;
    p.R = p.G + m;                       // rows of the expert products: the pairs, then the shared expert's m rows
    p.a0 = 0;
    p.r0 = (uint32_t) align16(p.a0 + 3 * p.GT * 8);
    p.w_off = (uint32_t) align16(p.r0 + 3 * p.GT * 17 * 4);
    p.counts_off = (uint32_t) align16(p.w_off + m * k * 4);
    p.tidx_off = (uint32_t) align16(p.counts_off + m * 4);
    p.bytes = (uint32_t) align16(p.tidx_off + m * k * 4);
    return p;
}

// An EXL3 layer's plan behind [tidx | w | cnt] (verify_plan_exl3 in kernels/exl3.hip): byte offset of the item list, item
// slots (a layer has at most one item a pair plus the shared expert's: the last slot is never an item), bytes of the whole.
struct VerifyPlan {
    uint32_t ioff, slots, bytes;
};
VerifyPlan verify_plan(uint32_t m, uint32_t k) {
    VerifyPlan p{};
    p.ioff = (uint32_t) align16(2ull * m * k * 4 + m * 4);
    p.slots = m * k + 2;
    p.bytes = p.ioff + 16 + p.slots * 32;
    return p;
}
// What the verify launches leave for one EXL3 layer: launch 2's sums (an f32 for every pair, projection, 512 inputs and ff
// column) and launch 3's.
uint64_t verify_part_bytes(const sz_session_config& c, uint32_t m) { return 2ull * m * (c.top_k + 1) * exl3_ksplit(c.hidden) * c.ff * 4; }
uint64_t verify_dn_bytes(const sz_session_config& c, uint32_t m) { return (uint64_t) m * (c.top_k + 1) * exl3_ksplit(c.ff) * c.hidden * 4; }

// The EXL3 layers table[p0 .. p1) for a batch of m rows: u, rl, sgl, y and `plans` are the caller's, layer `base`'s part first.
int verify_layers(sz_session* s, uint32_t p0, uint32_t p1, uint32_t base, uint32_t m, uint64_t u, uint64_t rl, uint64_t sgl, uint64_t y, uint64_t plans, uint64_t stream) {
    const sz_session_config& c = s->cfg;
    const VerifyPlan vp = verify_plan(m, c.top_k);
    const uint32_t zs = exl3_ksplit(c.hidden), zd = exl3_ksplit(c.ff);
    const bool one = p1 - p0 == 1;   // a single layer's addresses go along as kernel arguments, not through the table
    auto table = [&](uint32_t p) { return one ? 0 : s->vtab_dev.ptr + (uint64_t) p * sizeof(VerifyLayer); };
    const VerifyLayer& V = s->vtab[p0];
    if (one) {
        // its part of the buffers, wherever the caller's begin: without a table the kernels take it to be layer `base`, and without a
        // plan (below) they leave ids and weights at `plans` itself
        const uint64_t l = V.layer - base;
        u += l * m * c.hidden * 4;
        rl += l * m * c.n_expert * 4;
        sgl += l * m * 4;
        y += l * m * c.hidden * 4;
        plans += l * s->plan_stride;
        base = V.layer;
    }
    // Layer by layer, tokens that share an expert are worth a launch that finds them only where they are many: about 3 to 6 us
    // and a boundary, against the decode of a fifth of the pairs.  Measured a layer with and without the plan: 45 and 42 us at 4
    // rows of top-10 of 512 (distinct / pairs 0.97), 46.4 and 45.9 of top-8 of 128 (0.91), 68.7 and 70 of top-4 of 32 (0.83), 72
    // and 75 at 8 rows of top-8 of 128 (0.80), 104 and 128 of top-4 of 32 (0.66).  A round's plans are one launch for all layers.
    const double pairs = (double) m * c.top_k, distinct = c.n_expert * (1.0 - std::pow(1.0 - (double) c.top_k / c.n_expert, (double) m));
    const bool by_pair = one && distinct > 0.8 * pairs;
    const uint32_t ioff = by_pair ? 0 : vp.ioff, slots = by_pair ? m * c.top_k + 1 : vp.slots;
    if (!by_pair) {
        const sz_arg a[] = {P(rl), P(plans), U32(s->plan_stride), U32(vp.ioff), P(table(p0)), U64(V.shared), U32(base), U32(c.n_expert), U32(c.top_k), U32(m)};
        if (launch("verify_plan_exl3", p1 - p0, 1, 1, 64 * m, 0, stream, a)) return 1;
    }
    for (uint32_t q0 = p0; q0 < p1; q0 += s->vchunk) {
        const uint32_t q1 = std::min(p1, q0 + s->vchunk);
        for (uint32_t r0 = q0, r1; r0 < q1; r0 = r1) {   // runs of one type
            const int ty = s->layers[s->vtab[r0].layer].type;
            for (r1 = r0 + 1; r1 < q1 && s->layers[s->vtab[r1].layer].type == ty;) r1++;
            Format f;
            std::string tag;
            format_of(ty, f, tag);
            const uint32_t nl = r1 - r0;
            const uint64_t part = s->part.ptr + (r0 - q0) * verify_part_bytes(c, m), dn = s->dn.ptr + (r0 - q0) * verify_dn_bytes(c, m);
            uint32_t ct;
            {
                const std::string kn = std::string("verify_gate_up_") + verify_variant(c.ff, 2ull * nl * slots * zs * (c.ff / 128), m, &ct) + tag;
                const sz_arg a[] = {P(rl), P(table(r0)), U64(V.experts), U64(V.stride), U64(V.shared), U32(V.part), U32(base), P(plans), P(plans), U32(s->plan_stride), U32(ioff), P(u), P(part), U32(c.n_expert), U32(c.top_k),
                                    U32(m), U32(c.hidden), U32(c.ff)};
                if (launch(kn.c_str(), c.ff / (64 * ct), 2 * slots, nl * zs, 256, 0, stream, a)) return 1;
            }
            {
                const std::string kn = std::string(zs > 4 ? "verify_down_x_" : "verify_down_") + verify_variant(c.hidden, (uint64_t) nl * slots * zd * (c.hidden / 128), m, &ct) + tag;
                const sz_arg a[] = {P(rl), P(table(r0)), U64(V.experts), U64(V.stride), U64(V.shared), U32(V.part), U32(base), P(plans), P(plans), U32(s->plan_stride), U32(ioff), P(part), P(dn),
                                    U32(c.n_expert), U32(c.top_k), U32(m), U32(c.hidden), U32(c.ff)};
                if (launch(kn.c_str(), c.hidden / (64 * ct), slots, nl * zd, 256, 0, stream, a)) return 1;
            }
        }
        const sz_arg a[] = {P(s->dn.ptr), P(table(q0)), U64(V.experts), U64(V.stride), U64(V.shared), U32(V.part), U32(base), P(plans), U32(s->plan_stride), P(sgl), P(y), U32(c.top_k), U32(m), U32(c.hidden), U32(c.ff)};
        if (launch("verify_combine_exl3", c.hidden / 128, m, q1 - q0, 64 * std::min<uint32_t>(16, c.top_k + 1), 0, stream, a)) return 1;
    }
    return 0;
}

// The two launches of a single token (decode_gate_up_*, decode_down_combine_*): rows a workgroup and their LDS, if the shape has them.
struct DecodeShape {
    bool ok = false;
    uint32_t rp = 8, rd = 0, rs_gu = 0, rs_d = 0, pairs = 0;
};
DecodeShape decode_shape(const sz_session_config& c, const Format& f, bool shared) {
    DecodeShape d;
    const uint32_t uh = c.hidden / 32, uf = c.ff / 32;
    if (c.hidden % 32 || c.ff % 32 || uh > 64 || 64 % uh || uf > 64 || 64 % uf || c.top_k > 16) return d;
    d.rd = std::max(4u, 64 / uf);
    d.rs_gu = (d.rp * (c.hidden / f.qk * f.bb) + 31) / 16 * 16;
    d.rs_d = (d.rd * (c.ff / f.qk * f.bb) + 31) / 16 * 16;
    d.pairs = c.top_k + (shared ? 1 : 0);
    d.ok = c.ff % d.rp == 0 && c.hidden % d.rd == 0 && 2 * d.rs_gu <= 16384 && d.pairs * d.rs_d <= 16384 && d.pairs * c.ff <= 8192;
    return d;
}

// Whether a layer of GGUF experts runs on the matrix cores (verify_items) or the vector unit.  Their sums are in another order, and a
// token's bits must not depend on the other tokens of its batch (what a verify round accepts is what decoding token by token gives):
// the layer's shape alone decides, for one row to eight.  The more weights a token takes the sooner the matrix cores win; IQ3_S holds
// out longer where a single token has its two launches.  Measured, us of the router and the layer, four layers in a row, vector unit /
// matrix cores at 1, 2, 4 and 8 rows, by millions of weights a token:
//   Q8_0                       10.2: 17.9 20.3 28.7 43.1 / 19.2 23.0 31.1 53.2    11.0: 16.1 19.6 27.1 45.5 / 18.1 19.9 23.3 35.9
//                              18.9: 19.9 25.1 38.1 65.4 / 20.2 22.4 31.4 52.5    47.2: 30.6 54.2 93.0 167 / 25.2 36.0 59.6 88.5
//   IQ3_S with two launches    18.9: 17.6 25.5 30.9 50.7 / 20.8 23.9 33.4 57.1    34.6: 19.9 30.1 46.7 79.1 / 23.6 31.5 44.0 83.2
//                              40.9: 25.7 36.6 53.0 90.5 / 24.1 32.7 46.7 96.5    50.3: 28.6 40.1 63.2 108 / 24.8 33.4 54.3 80.4
//   IQ3_S without them         18.9: 20.2 24.2 36.4 59.5 / 22.3 24.3 36.5 57.5    20.6: 21.8 27.7 38.3 57.4 / 21.2 24.4 31.6 47.0
//                              47.2: 31.4 48.7 81.5 149 / 27.4 35.7 60.2 93.7
// A line in front of 34.6 would cost a single token a fifth; behind it layers of few experts lose what their tokens share (60 experts
// at 34.6: 19.8 29.7 45.6 73.9 / 23.7 31.4 43.3 57.9).  More than 4096 inputs of a down product are more than the vector kernels
// without a plan take; with one, 21.2 of Q8_0: 33.3 43.4 59.5 90.5 / 22.8 25.3 31.7 46.1.
bool gguf_matrix_cores(const sz_session_config& c, int type, const Format& f, bool shared) {
    if (c.ff > 4096) return true;
    const double weights = 3.0 * c.hidden * c.ff * (c.top_k + (shared ? 1 : 0));
    return weights >= (type == SZ_TYPE_Q8_0 ? 11e6 : decode_shape(c, f, shared).ok ? 40e6 : 20e6);
}

// A layer of GGUF experts by distinct expert on the matrix cores (verify_items_* in kernels/gguf.hip).
int verify_items(sz_session* s, const SzLayer& L, const std::string& tag, uint32_t m, uint64_t u, uint64_t rl, uint64_t sgl, uint64_t y, uint64_t plan, uint64_t stream) {
    const sz_session_config& c = s->cfg;
    Format f;
    std::string t;
    format_of(L.type, f, t);
    const uint64_t part = matrix_bytes(f, c.hidden, c.ff) + L.gap;   // from one projection of an expert to the next
    // The plan is a launch of 4.5 us: worth it where it saves the decode of about 30 M weights (expected, for independent choices); the bits
    // are the same either way.  Measured, us a layer with and without: 78.5 and 80.6 at 8 rows of top-10 of 512 Q8_0 experts of 2048 x 512
    // (17 M saved), 98.2 and 92.9 at 6 rows of top-8 of 256 of 3072 x 768 (25 M), 87.5 and 87.2 at 8 rows of top-8 of 128 of 2560 x 768 (73
    // M), 296 and 309 at 8 rows of top-12 of 512 of 3328 x 1536 (113 M), 55.6 and 85.5 at 8 rows of top-12 of 32 of 2048 x 512 (203 M): no
    // line has all of these right, the first takes 3 % more than it could here.
    const double pairs = (double) m * c.top_k, distinct = c.n_expert * (1.0 - std::pow(1.0 - (double) c.top_k / c.n_expert, (double) m));
    const char* form = std::getenv("SHADOWZERO_GGUF_ITEMS");
    const bool by_pair = form ? std::strcmp(form, "pairs") == 0 : (pairs - distinct) * 3.0 * c.hidden * c.ff < 30e6;
    const VerifyPlan vp = verify_plan(m, c.top_k);
    const uint32_t ioff = by_pair ? 0 : vp.ioff, ng = m > 4 ? 2 : 1;
    if (!by_pair) {
        const sz_arg a[] = {P(rl), P(plan), U32(s->plan_stride), U32(vp.ioff), P(0), U64(L.shared), U32(0), U32(c.n_expert), U32(c.top_k), U32(m)};
        if (launch("verify_plan_exl3", 1, 1, 1, 64 * m, 0, stream, a)) return 1;
    }
    // Row tiles a workgroup: more of them share the inputs' parts and a start worth about 5.5 tiles, fewer fill the chip.  Over 14
    // layers of both formats the choice is within 5 % of the best of 2, 4 and 8 (8 rows of top-8 of 128 Q8_0 experts of 2560 x 768: 100,
    // 88.1 and 87.5 us; 2 rows of top-10 of 512 IQ3_S experts of 2048 x 512: 33.3, 31.9 and 32.7).
    const double items = (by_pair ? pairs : distinct) + (L.shared ? 1 : 0);
    auto product = [&](const char* name, uint64_t in, uint64_t out, uint32_t tiles, uint32_t slots, uint32_t cols) {
        const uint32_t waves = gguf_waves(cols);
        uint32_t each = 0;
        double best = 1e30;
        for (uint32_t e = 8; e >= 2; e /= 2) {
            if (gguf_lds(waves, e, ng) > CU_LDS_BYTES - 4096) continue;
            const double cost = std::max(1.0, items * ((tiles + e - 1) / e) / (256 * (16 / waves))) * (e + 5.5);
            if (cost < best) best = cost, each = e;
        }
        const sz_arg a[] = {P(rl), U64(L.experts), U64(L.stride), U64(L.shared), U32((uint32_t) part), P(plan), U32(ioff), P(in), P(out), U32(c.n_expert), U32(c.top_k), U32(m),
                            U32(c.hidden), U32(c.ff)};
        return launch((name + std::string(m > 4 ? "w_" : "") + tag).c_str(), (tiles + each - 1) / each, slots, 1, 64 * waves, gguf_lds(waves, each, ng), stream, a);
    };
    // a slot past the items has the routing weights worked out: in the first launch behind a plan, else in the second
    if (product("verify_items_gate_up_", u, s->eg.ptr, 2 * c.ff / 16, m * c.top_k + (by_pair ? 1 : 2), c.hidden)) return 1;
    if (product("verify_items_down_", s->eg.ptr, s->eo.ptr, c.hidden / 16, m * c.top_k + (by_pair ? 2 : 1), c.ff)) return 1;
    s->last_fused = true;
    const uint64_t G4 = 4ull * m * c.top_k;
    const sz_arg a[] = {P(y), P(s->eo.ptr), P(plan + G4), P(L.shared ? s->eo.ptr + (uint64_t) m * c.top_k * c.hidden * 4 : 0), P(sgl), P(plan + 2 * G4), U32(c.hidden), U32(c.top_k)};
    return launch("moe_combine_qwen_rows", (c.hidden + 255) / 256, m, 1, 256, 0, stream, a);
}

int moe_layer(sz_session* s, uint32_t l, uint32_t m, uint64_t u, uint64_t rl, uint64_t sgl, uint64_t y, uint64_t stream) {
    const sz_session_config& c = s->cfg;
    if (l >= s->layers.size() || !s->layers[l].set) return fail("sz_moe_layer_verify: layer " + std::to_string(l) + " has no experts set");
    if (m == 0 || m > c.max_rows) return fail("sz_moe_layer_verify: " + std::to_string(m) + " rows (1.." + std::to_string(c.max_rows) + ")");
    if ((u & 15) || (y & 15)) return fail("sz_moe_layer_verify: activations must be 16-byte aligned");
    SzLayer& L = s->layers[l];
    Format f;
    std::string tag;
    if (!format_of(L.type, f, tag)) return fail("layer type " + std::to_string(L.type) + " has no kernels");
    const bool shared = L.shared != 0;
    if (shared && L.shared_type != L.type) return fail("the shared expert must have the routed experts' type (layer " + std::to_string(l) + ")");
    const PlanLayout p = plan_layout(m, c.top_k);
    const uint64_t plan = s->plan.ptr;
    s->last_plan = plan;
    if (f.exl3) {
        s->last_fused = true;
        return verify_layers(s, L.vpos, L.vpos + 1, l, m, u, rl, sgl, y, plan, stream);
    }
    const char* items = std::getenv("SHADOWZERO_GGUF_ITEMS");   // "plan" or "pairs": that form of the matrix cores at any size
    const bool apart = (matrix_bytes(f, c.hidden, c.ff) + L.gap) >> 32;   // projections further apart than these kernels' 32-bit offset reaches
    if ((items || gguf_matrix_cores(c, L.type, f, shared)) && !apart && !std::getenv("SHADOWZERO_GGUF_PLANNED")) return verify_items(s, L, tag, m, u, rl, sgl, y, plan, stream);
    const uint64_t addr = plan + p.a0, rec = plan + p.r0, wts = plan + p.w_off, cnt = plan + p.counts_off;
    const uint64_t addr_d = addr + 2ull * p.GT * 8, rec_d = rec + 2ull * p.GT * 17 * 4;
    const std::string kn = "matvec_grouped_" + tag;
    if (!std::getenv("SHADOWZERO_GGUF_PLANNED") && c.ff <= 4096) {
        // the pair form: routing inside launch 1, SwiGLU inside launch 2, no plan
        const uint32_t S = p.G + m;
        // (one row has few pairs to hand out: 16 and 32 rows a workgroup fill the chip better than 32 and 64, which win from two rows on: measured)
        const uint32_t rpb_gu = rows_per_block(f, c.hidden, m == 1 ? 16 : 32, m == 1 ? 16384 : 32768);
        const uint32_t rpb_d = rows_per_block(f, c.ff, m == 1 ? 32 : 64);
        if (!rpb_gu || !rpb_d) return fail("sz_moe_layer_verify: no kernel for hidden = " + std::to_string(c.hidden) + ", ff = " + std::to_string(c.ff));
        const uint64_t part = matrix_bytes(f, c.hidden, c.ff) + L.gap;   // from one projection of an expert to the next
        if (part >> 32) return fail("sz_moe_layer_verify: a projection of 4 GiB or more");
        const uint32_t rb_gu = c.hidden / f.qk * f.bb, rb_d = c.ff / f.qk * f.bb;
        // One token: two launches.  Launch 1 hands over act = silu(gate) * up and the routing weights, launch 2 owns a row chunk
        // for all of the token's experts and adds them up itself (SHADOWZERO_GGUF_THREE_LAUNCH=1 keeps the general form).
        const bool three = std::getenv("SHADOWZERO_GGUF_THREE_LAUNCH") != nullptr;
        const DecodeShape d = decode_shape(c, f, shared);
        if (m == 1 && !three && d.ok) {
            const std::string d1 = "decode_gate_up_" + tag, d2 = "decode_down_combine_" + tag;
            {
                const sz_arg a[] = {P(rl), U64(L.experts), U64(L.stride), U64(L.shared), U32((uint32_t) part), P(u), P(plan), P(s->eg.ptr),
                                    U32(c.n_expert), U32(c.top_k), U32(m), U32(c.hidden), U32(c.ff), U32(d.rp)};
                if (launch(d1.c_str(), c.ff / d.rp, S, 1, 512, 2 * d.rs_gu, stream, a)) return 1;   // 8 waves: a gate row and an up row each at hidden 2048
            }
            s->last_fused = true;
            const sz_arg a[] = {U64(L.experts), U64(L.stride), U64(L.shared), U32((uint32_t) part), P(plan), P(s->eg.ptr), P(sgl), P(y),
                                U32(c.top_k), U32(c.hidden), U32(c.ff), U32(d.rd)};
            return launch(d2.c_str(), c.hidden / d.rd, 1, 1, 64 * std::min(16u, std::max(4u, d.pairs)), d.pairs * d.rs_d + d.pairs * (c.ff / 32) * 144, stream, a);   // a wave a pair
        }
        const std::string k1 = "verify_gate_up_" + tag, k2 = "verify_down_" + tag;
        {
            const sz_arg a[] = {P(rl), U64(L.experts), U64(L.stride), U64(L.shared), U32((uint32_t) part), P(u), P(plan), P(s->eg.ptr),
                                U32(c.n_expert), U32(c.top_k), U32(m), U32(c.hidden), U32(c.ff), U32(rpb_gu)};
            if (launch(k1.c_str(), (c.ff + rpb_gu - 1) / rpb_gu, 2 * S, 1, 256, rpb_gu * rb_gu + 32, stream, a)) return 1;
        }
        {
            const sz_arg a[] = {P(rl), U64(L.experts), U64(L.stride), U64(L.shared), U32((uint32_t) part), P(plan), P(s->eg.ptr), P(s->eo.ptr),
                                U32(c.n_expert), U32(c.top_k), U32(m), U32(c.hidden), U32(c.ff), U32(rpb_d)};
            if (launch(k2.c_str(), (c.hidden + rpb_d - 1) / rpb_d, S, 1, 256, rpb_d * rb_d + 32, stream, a)) return 1;
        }
        s->last_fused = true;
        const uint64_t G4 = (uint64_t) p.G * 4;
        const sz_arg a[] = {P(y), P(s->eo.ptr), P(plan + G4), P(shared ? s->eo.ptr + (uint64_t) p.G * c.hidden * 4 : 0), P(sgl), P(plan + 2 * G4),
                            U32(c.hidden), U32(c.top_k)};
        return launch("moe_combine_qwen_rows", (c.hidden + 255) / 256, m, 1, 256, 0, stream, a);
    } else {
        {
            const sz_arg a[] = {P(rl), P(L.eaddr.ptr), P(plan), U32(c.n_expert), U32(c.top_k), U32(m), U32(p.G), U32(p.R), U32(p.a0), U32(p.r0),
                                U32(p.w_off), U32(p.counts_off), U32(p.tidx_off), P(shared ? L.eaddr.ptr + 3ull * c.n_expert * 8 : 0)};
            if (launch("route_plan_res_small", 1, 1, 1, 256, 0, stream, a)) return 1;
        }
        s->last_fused = false;
        const uint32_t rpb_gu = rows_per_block(f, c.hidden, std::max<uint32_t>(1, c.ff * 2 * p.GT / 512));
        const uint32_t rpb_d = rows_per_block(f, c.ff, std::max<uint32_t>(1, c.hidden * p.GT / 512));
        if (!rpb_gu || !rpb_d) return fail("this hidden / ff shape is not supported by the grouped " + tag + " kernels");
        const uint32_t rb_gu = c.hidden / f.qk * f.bb, rb_d = c.ff / f.qk * f.bb;
        {
            const sz_arg a[] = {P(addr), P(rec), P(u), U32(c.hidden), P(s->eg.ptr), U32(c.ff), U32(c.ff), U32(c.hidden), U32(rpb_gu)};
            if (launch(kn.c_str(), (c.ff + rpb_gu - 1) / rpb_gu, 2 * p.GT, 1, 256, rpb_gu * rb_gu + 32, stream, a)) return 1;
        }
        {
            const uint32_t n = p.R * c.ff;
            const sz_arg a[] = {P(s->eg.ptr), P(s->eg.ptr + (uint64_t) p.R * c.ff * 4), P(s->act.ptr), U32(n)};
            if (launch("swiglu", (n + 255) / 256, 1, 1, 256, 0, stream, a)) return 1;
        }
        {
            const sz_arg a[] = {P(addr_d), P(rec_d), P(s->act.ptr), U32(c.ff), P(s->eo.ptr), U32(c.hidden), U32(c.hidden), U32(c.ff), U32(rpb_d)};
            if (launch(kn.c_str(), (c.hidden + rpb_d - 1) / rpb_d, p.GT, 1, 256, rpb_d * rb_d + 32, stream, a)) return 1;
        }
    }
    const sz_arg a[] = {P(y), P(s->eo.ptr), P(wts), P(shared ? s->eo.ptr + (uint64_t) p.G * c.hidden * 4 : 0), P(sgl), P(cnt), U32(c.hidden), U32(c.top_k)};
    return launch("moe_combine_qwen_rows", (c.hidden + 255) / 256, m, 1, 256, 0, stream, a);
}

// The head for rows [j0, j0 + n) with the arg-max fused in; logits (0: not written) has rows c.vocab apart.
int head_argmax_rows(sz_session* s, uint32_t n, uint64_t u, uint64_t logits, uint64_t ids, uint64_t stream) {
    const sz_session_config& c = s->cfg;
    Format f;
    std::string tag;
    format_of(s->head_type, f, tag);
    const uint32_t rpb = rows_per_block(f, c.hidden);
    if (!rpb) return fail("the head kernel does not support hidden = " + std::to_string(c.hidden));
    const uint32_t rb = c.hidden / 32 * 34, nchunks = (c.vocab + rpb - 1) / rpb;
    const uint32_t nparts = std::min<uint32_t>(nchunks, persistent_groups());
    const sz_arg a[] = {P(s->head_w), P(u), U32(c.hidden), P(logits), U32(c.vocab), P(s->head_part.ptr), U32(c.vocab), U32(c.hidden), U32(n), U32(rpb)};
    if (launch("head_q8_0_argmax", nparts, 1, 1, 256, rpb * rb + 32 + rpb * 16, stream, a)) return 1;
    const sz_arg b[] = {P(s->head_part.ptr), U32(nparts), U32(4), P(ids), P(0)};
    return launch("argmax_merge_parts", n, 1, 1, 256, 0, stream, b);
}

// The end of a head pass: the rows' arg-max ids out of the partial maxima; with `accept` set (a verify round), the greedy
// acceptance of the drafts in the same launch.
struct Accept {
    uint64_t drafts = 0, out = 0;
};
int merge_parts(sz_session* s, uint32_t nparts, uint32_t ts, uint32_t m, uint64_t ids, const Accept* accept, uint64_t stream) {
    if (accept) {
        const sz_arg a[] = {P(s->head_part.ptr), U32(nparts), U32(ts), P(ids), U32(m), P(accept->drafts), U32(m - 1), P(accept->out)};
        return launch("argmax_merge_accept", 1, 1, 1, 1024, 0, stream, a);
    }
    const sz_arg b[] = {P(s->head_part.ptr), U32(nparts), U32(ts), P(ids), P(0)};
    return launch("argmax_merge_parts", m, 1, 1, 256, 0, stream, b);
}

// The matrix-core head: all m <= 8 rows in one pass over the matrix.  The number of waves a workgroup (each owns at most
// 512 columns of a row): 4 up to 2048 columns, 6 up to 3072, 8 up to 4096; 0: the shape goes to the scalar kernel.
uint32_t head_mfma_waves(const sz_session* s) {
    static const bool off = std::getenv("SHADOWZERO_HEAD_SCALAR") != nullptr;
    const sz_session_config& c = s->cfg;
    if (off || s->head_type != SZ_TYPE_Q8_0 || (s->head_w & 15) != 0 || c.vocab < 16) return 0;
    if (c.hidden % 256 == 0 && c.hidden <= 2048) return 4;
    if (c.hidden % 192 == 0 && c.hidden <= 3072) return 6;
    if (c.hidden % 256 == 0 && c.hidden <= 4096) return 8;
    return 0;
}
bool head_mfma_ok(const sz_session* s) { return head_mfma_waves(s) != 0; }

int head_argmax_mfma(sz_session* s, uint32_t m, uint64_t u, uint64_t logits, uint64_t ids, uint64_t stream, const Accept* accept = nullptr) {
    const sz_session_config& c = s->cfg;
    const uint32_t waves = head_mfma_waves(s);
    const uint32_t tiles = (c.vocab + 15) / 16;
    const uint32_t nparts = std::min<uint32_t>(tiles, waves == 4 ? 512 : 256);       // two workgroups a CU (70 KB of LDS each), one for the wider rows
    const sz_arg a[] = {P(s->head_w), P(u), U32(c.hidden), P(logits), U32(c.vocab), P(s->head_part.ptr), U32(c.vocab), U32(c.hidden), U32(m)};
    const char* name = waves == 4 ? "head_q8_0_argmax_mfma" : waves == 6 ? "head_q8_0_argmax_mfma_w6" : "head_q8_0_argmax_mfma_w8";
    static const bool four_waves = std::getenv("SHADOWZERO_HEAD_FOUR_WAVES") != nullptr;   // the general form at 2048 columns too, for comparisons
    if (waves == 4 && c.hidden == 2048 && !four_waves) {
        // rows of exactly 2048 columns: 8 waves of 256 columns each on the same two tiles of LDS, no per-block checks
        if (launch("head_q8_0_argmax_mfma_n8", nparts, 1, 1, 512, 0, stream, a)) return 1;
        return merge_parts(s, nparts, 8, m, ids, accept, stream);
    }
    if (launch(name, nparts, 1, 1, 64 * waves, 0, stream, a)) return 1;
    return merge_parts(s, nparts, 8, m, ids, accept, stream);
}

bool head_is_exl3(const sz_session* s) { return s->head_type >= 1021 && s->head_type <= 1028; }

// The rows a call of an EXL3 head may bring are a limit of this interface, which callers size their batches by (sz_exl3_head_lds_bytes
// against CU_LDS_BYTES): the LDS of a workgroup that keeps its A rows there, four 4-row rings (a row is 64 lanes x 4 words at K = 3 and
// 4, x K words otherwise) and 4 KiB for every 512 inputs and every two rows.  head_exl3_K itself takes 24 KiB whatever the rows.
uint32_t exl3_head_lds(uint32_t bits, uint32_t hidden, uint32_t m) {
    const uint32_t stride = (bits == 3 || bits == 4) ? 4 : bits;
    return 4 * (4 * 64 * stride) * 4 + 4 * ((hidden / 128 + 3) / 4) * ((m + 1) / 2) * 1024;
}

int head_check(sz_session* s, uint32_t m, uint64_t u, const char* who) {
    if (!s->head_w) return fail(std::string(who) + ": no head set");
    if (m == 0 || m > s->cfg.max_rows) return fail(std::string(who) + ": " + std::to_string(m) + " rows");
    if (u & 15) return fail(std::string(who) + ": activations must be 16-byte aligned");
    if (head_is_exl3(s) && exl3_head_lds((uint32_t) s->head_type - 1020, s->cfg.hidden, m) > CU_LDS_BYTES)
        return fail(std::string(who) + ": " + std::to_string(m) + " rows are above the limit of an EXL3 head of hidden " + std::to_string(s->cfg.hidden) + " at " +
                    std::to_string(s->head_type - 1020) + " bits (sz_exl3_head_lds_bytes above " + std::to_string(CU_LDS_BYTES) + "): fewer rows a call");
    return 0;
}

// Q8_0 and EXL3 heads have the arg-max fused into the product; every other type goes through its logits (set_head keeps the
// buffer for them).
bool head_argmax_fused(const sz_session* s) { return s->head_type == SZ_TYPE_Q8_0 || head_is_exl3(s); }

// The product launch of an EXL3 head over n output blocks (sel: a list of them, 0: all).  A head of more than 256 MiB, what the last level holds, is read past
// the caches (384 MiB at 6 bits, us of a round of 1 and 4 layers for one row 122 -> 118, 135 -> 132; 297 MiB at 4 bits 124 -> 121, 151 -> 149).  A smaller one is there
// again at the next call, also with layers in between (past the caches rounds of 1, 4 and 16 layers for four rows with 223 MiB 96 -> 102, 134 -> 136, 245 -> 255,
// with 111 MiB 89 -> 90, 125 -> 127, 231 -> 234, of 48 layers 1 % either way; a call alone with 223 MiB 79 -> 83; one that finds none of its 148 MiB 75.2 -> 74.0).
// A list's blocks are few.
int head_exl3_blocks(sz_session* s, uint32_t n, uint32_t m, uint64_t logits, uint32_t ls, uint64_t sel, uint64_t stream) {
    const sz_session_config& c = s->cfg;
    const sz_arg a[] = {P(s->head_w), P(s->head_xa.ptr), P(s->head_inv.ptr), P(logits), U32(ls), P(s->head_part.ptr), U32(c.hidden), U32(c.vocab), U32(m), P(sel)};
    const uint32_t bits = (uint32_t) s->head_type - 1020;
    const bool past = !sel && (uint64_t) c.hidden * c.vocab * bits / 8 > 256ull << 20;
    return launch(((past ? "head_exl3_past_" : "head_exl3_") + std::to_string(bits)).c_str(), n, 1, 1, 256, 0, stream, a);
}

// An EXL3 head (kernels/exl3.cu:349-461, 610-625 of the reference: rotate the rows once, then one pass over the matrix for all
// m <= 8 rows): the arg-max ids (0: not wanted) and / or the logits (0: not written).
int head_exl3(sz_session* s, uint32_t m, uint64_t u, uint64_t logits, uint64_t ids, uint64_t stream, const Accept* accept = nullptr) {
    const sz_session_config& c = s->cfg;
    const uint32_t kbs = c.hidden / 128;
    {
        const sz_arg a[] = {P(s->head_w), P(u), U32(c.hidden), P(s->head_xa.ptr), P(s->head_inv.ptr), U32(c.hidden)};
        if (launch("exl3_head_rotate", m, 1, 1, 64 * std::min<uint32_t>(16, kbs), 0, stream, a)) return 1;
    }
    const uint32_t nparts = c.vocab / 128;
    if (head_exl3_blocks(s, nparts, m, logits, c.vocab, 0, stream)) return 1;
    if (!ids) return 0;
    return merge_parts(s, nparts, 8, m, ids, accept, stream);
}

// The number of blocks a row may choose for a hand-off of need_k values (session.rs:5961): three quarters of k_blk, at least
// 64, when only a few are needed.
uint32_t head_proxy_k_use(const sz_session* s, uint32_t need_k) {
    const uint32_t k = s->hp.k_blk;
    return need_k <= 16 ? std::min(std::max(k * 3 / 4, 64u), k) : k;
}

// The screened head (mv_head_proxy_sparse, session.rs:5952-5995): rotate the rows, their int8 codes, the block maxima of the
// 2-bit copy, the k_use best blocks of every row, their union as a list, and the exact head on the listed blocks only.
// Leaves the list in hp.sel and the packed logits (rows max_sel * 128 apart) in hp.logits; *max_sel_out = the list's bound.
int head_proxy_sparse(sz_session* s, uint32_t m, uint64_t u, uint32_t need_k, uint32_t* max_sel_out, uint64_t stream) {
    const sz_session_config& c = s->cfg;
    const uint32_t kbs = c.hidden / 128, n_ob = c.vocab / 128;
    const uint32_t k_use = head_proxy_k_use(s, need_k), max_sel = std::min(m * k_use, n_ob);
    {
        const sz_arg a[] = {P(s->head_w), P(u), U32(c.hidden), P(s->head_xa.ptr), P(s->head_inv.ptr), U32(c.hidden)};
        if (launch("exl3_head_rotate", m, 1, 1, 64 * std::min<uint32_t>(16, kbs), 0, stream, a)) return 1;
    }
    {
        const sz_arg a[] = {P(s->head_w), P(u), U32(c.hidden), P(s->hp.xq.ptr), P(s->hp.x_sc.ptr), P(s->hp.x_corr.ptr), U32(c.hidden)};
        if (launch("proxy_q2_quant_x", kbs, m, 1, 64, 0, stream, a)) return 1;
    }
    {
        const sz_arg a[] = {P(s->hp.w_q2.ptr), P(s->hp.w_sc.ptr), P(s->hp.xq.ptr), P(s->hp.x_sc.ptr), P(s->hp.x_corr.ptr), P(s->hp.bmax.ptr),
                            U32(n_ob), U32(c.hidden), U32(m)};
        if (launch(m == 1 ? "proxy_q2_bmax_m1" : m <= 4 ? "proxy_q2_bmax_m4" : "proxy_q2_bmax_m8", n_ob, 1, 1, 128, 0, stream, a)) return 1;
    }
    {
        const sz_arg a[] = {P(s->hp.bmax.ptr), U32(n_ob), U32(k_use), P(s->hp.seen.ptr)};
        if (launch("proxy_pick_rows", m, 1, 1, 1024, 0, stream, a)) return 1;
    }
    {
        const sz_arg a[] = {P(s->hp.seen.ptr), U32(n_ob), U32(max_sel), P(s->hp.sel.ptr)};
        if (launch("proxy_compact_seen", 1, 1, 1, 64, 0, stream, a)) return 1;
    }
    if (head_exl3_blocks(s, max_sel, m, s->hp.logits.ptr, max_sel * 128, s->hp.sel.ptr, stream)) return 1;
    *max_sel_out = max_sel;
    return 0;
}

int head_logits(sz_session* s, uint32_t m, uint64_t u, uint64_t logits, uint64_t stream);

// accept (a verify round): the greedy acceptance after the ids, fused into the merge where the head has one merge for all rows
int head_argmax(sz_session* s, uint32_t m, uint64_t u, uint64_t ids, uint64_t stream, const Accept* accept = nullptr) {
    if (head_check(s, m, u, "sz_head_argmax")) return 1;
    if (!head_argmax_fused(s)) {
        // mv_cols + topk_rows_at (session.rs:7034-7052): the logits, the largest of every slice of 4096, the largest of those
        const sz_session_config& c = s->cfg;
        const uint32_t nparts = (c.vocab + 4095) / 4096;
        if (head_logits(s, m, u, s->logits.ptr, stream)) return 1;
        const sz_arg a[] = {P(s->logits.ptr), U32(c.vocab), U32(c.vocab), P(s->head_part.ptr), U32(8)};
        if (launch("argmax_slices", nparts, m, 1, 256, 0, stream, a)) return 1;
        return merge_parts(s, nparts, 8, m, ids, accept, stream);
    }
    if (head_is_exl3(s)) return head_exl3(s, m, u, 0, ids, stream, accept);
    if (head_mfma_ok(s)) return head_argmax_mfma(s, m, u, 0, ids, stream, accept);
    for (uint32_t j0 = 0; j0 < m; j0 += 4) {
        if (head_argmax_rows(s, std::min(4u, m - j0), u + (uint64_t) j0 * s->cfg.hidden * 4, 0, ids + j0 * 4ull, stream)) return 1;
    }
    if (accept) {   // the scalar head merges four rows at a time: the acceptance is a launch of its own
        const sz_arg a[] = {P(ids), P(accept->drafts), U32(m - 1), P(accept->out)};
        return launch("verify_accept", 1, 1, 1, 64, 0, stream, a);
    }
    return 0;
}

int head_logits(sz_session* s, uint32_t m, uint64_t u, uint64_t logits, uint64_t stream) {
    if (head_check(s, m, u, "sz_head_logits")) return 1;
    if (head_is_exl3(s)) return head_exl3(s, m, u, logits, 0, stream);
    if (head_mfma_ok(s)) return head_argmax_mfma(s, m, u, logits, s->ids.ptr, stream);   // one pass for all rows; the ids are a by-product
    const sz_session_config& c = s->cfg;
    return matvec_cols_dev(s->head_type, s->head_w, c.hidden, c.vocab, u, c.hidden, logits, c.vocab, m, 0, 0, stream);
}

}   // namespace

extern "C" {

sz_session* sz_session_new(const sz_session_config* cfg) {
    clear_error();
    if (ensure_init()) return nullptr;
    const sz_session_config& c = *cfg;
    if (c.hidden == 0 || c.hidden % 256 || c.ff == 0 || c.ff % 256) { fail("sz_session_new: hidden and ff must be multiples of 256"); return nullptr; }
    if (c.n_expert == 0 || c.n_expert > 512 || c.top_k == 0 || c.top_k > 16 || c.max_rows == 0 || c.max_rows > 8) {
        fail("sz_session_new: needs n_expert <= 512, top_k <= 16, max_rows <= 8");   // the planner's limits (session.rs:8190-8202)
        return nullptr;
    }
    sz_session* s = new sz_session();
    s->cfg = c;
    s->layers.resize(c.n_layers);
    const PlanLayout p = plan_layout(c.max_rows, c.top_k);
    s->GT_max = p.GT;
    const uint64_t nparts = c.vocab / 4 + 1;
    s->plan_stride = (verify_plan(c.max_rows, c.top_k).bytes + 255) & ~255u;
    bool bad = s->plan.need(std::max(p.bytes, s->plan_stride)) || s->eg.need(2ull * p.R * c.ff * 4) || s->act.need((uint64_t) p.R * c.ff * 4) ||
               s->eo.need((uint64_t) p.R * c.hidden * 4) || s->ids.need(64);
    if (c.vocab) bad = bad || s->head_part.need(nparts * 4 * 2 * 4);
    if (bad) {
        delete s;
        return nullptr;
    }
    return s;
}

void sz_session_free(sz_session* s) {
    if (!s) return;
    if (s->top_host) hip().hipHostFree(s->top_host);
    for (auto& g : s->graphs) sz_graph_destroy(g.second.exec);
    delete s;
}

// The table of the EXL3 layers that are set, rebuilt and copied to the device.  (After a failed copy the caller unsets its layer:
// rounds, which alone read the device's copy, are refused until a later call has made it whole.)
static int verify_table(sz_session* s) {
    std::vector<uint32_t> order;
    for (uint32_t l = 0; l < s->layers.size(); l++)
        if (s->layers[l].set && s->layers[l].type > 1020) order.push_back(l);
    std::stable_sort(order.begin(), order.end(), [&](uint32_t a, uint32_t b) { return s->layers[a].type < s->layers[b].type; });
    s->vtab.clear();
    for (uint32_t l : order) {
        SzLayer& L = s->layers[l];
        Format f;
        std::string tag;
        format_of(L.type, f, tag);
        L.vpos = (uint32_t) s->vtab.size();
        s->vtab.push_back({L.experts, L.stride, L.shared, (uint32_t) (matrix_bytes(f, s->cfg.hidden, s->cfg.ff) + L.gap), l});
    }
    return s->vtab.empty() ? 0 : sz_upload(s->vtab_dev.ptr, s->vtab.data(), s->vtab.size() * sizeof(VerifyLayer));
}

int32_t sz_session_set_layer_spaced(sz_session* s, uint32_t l, int32_t ty, uint64_t experts, uint64_t stride, uint64_t gap, int32_t shared_type, uint64_t shared) {
    clear_error();
    if (!s || l >= s->layers.size()) return fail("sz_session_set_layer: no layer " + std::to_string(l));
    Format f;
    std::string tag;
    if (!format_of(ty, f, tag)) return fail("sz_session_set_layer: ggml type " + std::to_string(ty) + " has no kernels");
    const sz_session_config& c = s->cfg;
    const uint64_t gu = matrix_bytes(f, c.hidden, c.ff) + gap, dn = matrix_bytes(f, c.ff, c.hidden);   // gu: from a projection to the next
    if (stride < 2 * gu + dn) return fail("sz_session_set_layer: the expert stride is smaller than an expert");
    if ((experts | stride | shared | gap) & 3) return fail("sz_session_set_layer: expert blobs must be 4-byte aligned");
    if (gu >> 32) return fail("sz_session_set_layer: a projection of 4 GiB or more");
    SzLayer& L = s->layers[l];
    // the address table eaddr[part * ne + e] (session.rs:2129-2146), then the shared expert's three parts
    std::vector<uint64_t> tab(3ull * c.n_expert + 3);
    for (uint32_t e = 0; e < c.n_expert; e++) {
        const uint64_t b = experts + e * stride;
        tab[e] = b;
        tab[c.n_expert + e] = b + gu;
        tab[2ull * c.n_expert + e] = b + 2 * gu;
    }
    Format fs;
    std::string tags;
    if (shared) {
        if (!format_of(shared_type, fs, tags)) return fail("sz_session_set_layer: shared type " + std::to_string(shared_type) + " has no kernels");
        const uint64_t sgu = matrix_bytes(fs, c.hidden, c.ff) + gap;
        tab[3ull * c.n_expert] = shared;
        tab[3ull * c.n_expert + 1] = shared + sgu;
        tab[3ull * c.n_expert + 2] = shared + 2 * sgu;
    }
    // the allocations first: one that fails leaves the layer as it was
    if (f.exl3) {
        // the launches' buffers hold as many layers as take 256 MiB (what the memory-side cache holds), at least one
        const uint64_t per = verify_part_bytes(c, c.max_rows) + verify_dn_bytes(c, c.max_rows);
        s->vchunk = (uint32_t) std::min<uint64_t>(c.n_layers, std::max<uint64_t>(1, (256ull << 20) / per));
        if (s->plans.need((uint64_t) c.n_layers * s->plan_stride) || s->vtab_dev.need(c.n_layers * sizeof(VerifyLayer)) ||
            s->part.need(s->vchunk * verify_part_bytes(c, c.max_rows)) || s->dn.need(s->vchunk * verify_dn_bytes(c, c.max_rows)))
            return 1;
    }
    if (L.eaddr.need(tab.size() * 8)) return 1;
    // then the copies: the layer is unset while one of its tables may be half written
    L.set = false;
    if (sz_upload(L.eaddr.ptr, tab.data(), tab.size() * 8)) return 1;
    L.type = ty;
    L.shared_type = shared_type;
    L.experts = experts;
    L.stride = stride;
    L.shared = shared;
    L.gap = gap;
    L.set = true;
    if (verify_table(s)) {
        L.set = false;
        return 1;
    }
    for (auto& g : s->graphs) sz_graph_destroy(g.second.exec);   // captured address tables may be stale
    s->graphs.clear();
    return 0;
}

int32_t sz_session_set_layer(sz_session* s, uint32_t l, int32_t ty, uint64_t experts, uint64_t stride, int32_t shared_type, uint64_t shared) {
    return sz_session_set_layer_spaced(s, l, ty, experts, stride, 0, shared_type, shared);
}

// Where a layer's experts should lie for their rows to start on 128-byte lines of memory.  An EXL3 projection's trellis
// begins 2 (in + out) + 4 bytes into its blob (exl3.rs:390-393), and a launch fetches a row of it in segments of 512 to
// 2048 bytes: 4 bytes off a line, every segment touches one line more than it fills.  With the first blob `lead` bytes past
// a 128-byte boundary, `gap` bytes between an expert's projections and a stride that is a multiple of 128, every trellis
// starts on a line.  GGUF rows (34- and 110-byte blocks) have no such boundary: lead and gap 0.
void sz_layer_spacing(int32_t ty, uint64_t hidden, uint64_t ff, uint32_t* lead, uint32_t* gap) {
    Format f;
    std::string tag;
    uint32_t ld = 0, gp = 0;
    if (format_of(ty, f, tag) && f.exl3) {
        ld = (uint32_t) ((128 - (2 * (hidden + ff) + 4) % 128) % 128);
        gp = (uint32_t) ((128 - matrix_bytes(f, hidden, ff) % 128) % 128);
    }
    if (lead) *lead = ld;
    if (gap) *gap = gp;
}

int32_t sz_session_set_router(sz_session* s, uint32_t l, int32_t rty, uint64_t rw, int32_t gty, uint64_t gw) {
    clear_error();
    if (!s || l >= s->layers.size()) return fail("sz_session_set_router: no layer " + std::to_string(l));
    const sz_session_config& c = s->cfg;
    Format fr, fg;
    std::string tr, tg;
    if (!format_of(rty, fr, tr) || !fr.dense) return fail("sz_session_set_router: the router must be F32, F16 or BF16");
    if (gw && (!format_of(gty, fg, tg) || !fg.dense)) return fail("sz_session_set_router: the shared expert's gate must be F32, F16 or BF16");
    if (!rw || (rw & (4 * fr.bb - 1)) || (gw & (4 * (gw ? fg.bb : 1) - 1))) return fail("sz_session_set_router: matrices must be aligned to four weights");
    if (s->rl.need((uint64_t) c.max_rows * c.n_expert * 4) || s->sgl.need((uint64_t) c.max_rows * 4)) return 1;
    SzLayer& L = s->layers[l];
    L.router = rw;
    L.router_type = rty;
    L.gate = gw;
    L.gate_type = gty;
    for (auto& g : s->graphs) sz_graph_destroy(g.second.exec);
    s->graphs.clear();
    return 0;
}

int32_t sz_moe_router_verify(sz_session* s, uint32_t l, uint32_t m, uint64_t u, uint64_t stream) {
    clear_error();
    if (!s || l >= s->layers.size() || !s->layers[l].router) return fail("sz_moe_router_verify: layer " + std::to_string(l) + " has no router set");
    const sz_session_config& c = s->cfg;
    if (m == 0 || m > c.max_rows) return fail("sz_moe_router_verify: " + std::to_string(m) + " rows (1.." + std::to_string(c.max_rows) + ")");
    if (u & 15) return fail("sz_moe_router_verify: activations must be 16-byte aligned");
    const SzLayer& L = s->layers[l];
    const DenseShape d = dense_shape(c.hidden);
    const sz_arg a[] = {U32(dense_code(L.router_type)), P(L.router), U32(dense_code(L.gate_type)), P(L.gate), P(u), P(s->rl.ptr), P(s->sgl.ptr),
                        U32(c.n_expert), U32(c.hidden), U32(m)};
    return launch((std::string("router_rows_m") + dense_m(m)).c_str(), (c.n_expert + d.pass - 1) / d.pass + (L.gate ? 1 : 0), 1, 1, d.block, 0, stream, a);
}

int32_t sz_session_router_outputs(sz_session* s, uint64_t* rl, uint64_t* sgl) {
    clear_error();
    if (!s || !s->rl.ptr) return fail("sz_session_router_outputs: no router set");
    *rl = s->rl.ptr;
    *sgl = s->sgl.ptr;
    return 0;
}

int32_t sz_moe_block_verify(sz_session* s, uint32_t l, uint32_t m, uint64_t u, uint64_t y, uint64_t stream) {
    if (sz_moe_router_verify(s, l, m, u, stream)) return 1;
    return moe_layer(s, l, m, u, s->rl.ptr, s->sgl.ptr, y, stream);
}

int32_t sz_session_set_head(sz_session* s, int32_t ty, uint64_t w) {
    clear_error();
    if (!s) return fail("sz_session_set_head: null session");
    const bool exl3 = ty >= 1021 && ty <= 1028;
    const bool plain = ty == SZ_TYPE_F32 || ty == SZ_TYPE_F16 || ty == SZ_TYPE_BF16;
    if (ty != SZ_TYPE_Q8_0 && ty != SZ_TYPE_IQ3_S && !plain && !exl3)
        return fail("sz_session_set_head: the head must be Q8_0, IQ3_S, F32, F16, BF16 or EXL3 at a whole bit rate");
    // a type without a fused arg-max keeps its logits: allocated here, never during a call (a call may be under capture)
    if (ty != SZ_TYPE_Q8_0 && !exl3 && s->logits.need((uint64_t) s->cfg.max_rows * s->cfg.vocab * 4)) return 1;
    if (w & 15) return fail("sz_session_set_head: the head must be 16-byte aligned");
    if (exl3) {
        const sz_session_config& c = s->cfg;
        if (c.vocab == 0 || c.vocab % 128 || c.hidden % 128 || c.hidden > 8192) return fail("sz_session_set_head: an EXL3 head needs hidden (<= 8192) and the vocabulary to be multiples of 128");
        // one row is within the limit of every such head; how many a call may bring is checked call by call
        if (s->head_xa.need((uint64_t) c.hidden / 128 * 16 * 256) || s->head_inv.need(64)) return 1;
    }
    s->head_type = ty;
    s->head_w = w;
    s->hp.k_blk = 0;   // a screen belongs to the head it was built from
    for (auto& g : s->graphs) sz_graph_destroy(g.second.exec);
    s->graphs.clear();
    return 0;
}

uint32_t sz_exl3_head_lds_bytes(int32_t ty, uint32_t hidden, uint32_t m) {
    return (ty >= 1021 && ty <= 1028) ? exl3_head_lds((uint32_t) ty - 1020, hidden, m) : 0;
}

int32_t sz_session_set_head_proxy(sz_session* s, uint32_t k_blk) {
    clear_error();
    if (!s) return fail("sz_session_set_head_proxy: null session");
    if (k_blk == 0) {
        s->hp.k_blk = 0;
        return 0;
    }
    const sz_session_config& c = s->cfg;
    if (!head_is_exl3(s)) return fail("sz_session_set_head_proxy: the screen is built from an EXL3 head (set one first)");
    if (c.hidden > 4096) return fail("sz_session_set_head_proxy: hidden above 4096");      // session.rs:2656
    const uint64_t n_ob = c.vocab / 128, n_b = c.hidden / 128, rows = 8;
    const uint32_t k = (uint32_t) std::min<uint64_t>(std::max<uint32_t>(k_blk, 16), n_ob);   // session.rs:2659
    const uint64_t max_sel = std::min<uint64_t>(rows * k, n_ob);
    if ((max_sel * 128 + 4095) / 4096 > 64) return fail("sz_session_set_head_proxy: 8 rows of k_blk blocks are more than the top-64 merge takes (k_blk <= 256)");
    auto& h = s->hp;
    if (h.w_q2.need((uint64_t) c.vocab * c.hidden / 4) || h.w_sc.need((uint64_t) c.vocab * n_b * 2) || h.xq.need(rows * n_b * 32 * 4) ||
        h.x_sc.need(rows * n_b * 4) || h.x_corr.need(rows * n_b * 4) || h.bmax.need(rows * n_ob * 4) || h.seen.need((n_ob + 31) / 32 * 4) ||
        h.sel.need((1 + max_sel) * 4) || h.logits.need(rows * max_sel * 128 * 4))
        return 1;
    if (sz_memset(h.seen.ptr, 0, h.seen.bytes, 0) || sz_memset(h.xq.ptr, 0, h.xq.bytes, 0) || sz_memset(h.x_sc.ptr, 0, h.x_sc.bytes, 0) ||
        sz_memset(h.x_corr.ptr, 0, h.x_corr.bytes, 0))
        return 1;
    const std::string kn = "exl3_build_q2_proxy_" + std::to_string(s->head_type - 1020);
    const sz_arg a[] = {P(s->head_w), P(h.w_q2.ptr), P(h.w_sc.ptr), U32(c.hidden), U32(c.vocab)};
    if (launch(kn.c_str(), (uint32_t) n_ob, (uint32_t) n_b, 1, 256, 0, 0, a)) return 1;
    if (sz_stream_synchronize(0)) return 1;
    h.k_blk = k;
    return 0;
}

uint64_t sz_session_buffer(sz_session* s, int32_t which) {
    if (!s) return 0;
    const uint64_t at[] = {s->last_plan ? s->last_plan : s->plan.ptr, s->part.ptr, s->dn.ptr, s->eg.ptr, s->eo.ptr, s->hp.w_q2.ptr, s->hp.w_sc.ptr, s->hp.xq.ptr, s->hp.x_sc.ptr,
                           s->hp.x_corr.ptr, s->hp.bmax.ptr, s->hp.sel.ptr, s->hp.logits.ptr, s->pf.arows.ptr, s->pf.eo.ptr, s->pf.drows.ptr, s->pf.dinv.ptr, s->pf.items.ptr};
    return which >= 0 && which < (int32_t) (sizeof at / sizeof at[0]) ? at[which] : 0;
}

int32_t sz_session_set_expert_mode(sz_session* s, int32_t mode) {
    clear_error();
    if (!s) return fail("sz_session_set_expert_mode: null session");
    if (mode < 0 || mode > 3)
        return fail("sz_session_set_expert_mode: mode " + std::to_string(mode) + " (0 to 3)");
    return 0;
}

int32_t sz_session_set_graph(sz_session* s, int32_t enabled) {
    clear_error();
    if (!s) return fail("sz_session_set_graph: null session");
    s->use_graph = enabled != 0;
    return 0;
}

int32_t sz_moe_layer_verify(sz_session* s, uint32_t l, uint32_t m, uint64_t u, uint64_t rl, uint64_t sgl, uint64_t y, uint64_t stream) {
    clear_error();
    if (!s) return fail("sz_moe_layer_verify: null session");
    return moe_layer(s, l, m, u, rl, sgl, y, stream);
}

int32_t sz_session_last_route(sz_session* s, uint32_t m, uint32_t* idx, float* w, uint64_t stream) {
    clear_error();
    if (!s || m == 0 || m > s->cfg.max_rows) return fail("sz_session_last_route: bad arguments");
    if (sz_stream_synchronize(stream)) return 1;
    const PlanLayout p = plan_layout(m, s->cfg.top_k);
    const uint64_t n = (uint64_t) m * s->cfg.top_k * 4;
    const uint64_t plan = s->last_plan ? s->last_plan : s->plan.ptr;
    if (s->last_fused) return sz_download(idx, plan, n) || sz_download(w, plan + n, n);
    if (sz_download(idx, plan + p.tidx_off, n)) return 1;
    return sz_download(w, plan + p.w_off, n);
}

int32_t sz_head_argmax(sz_session* s, uint32_t m, uint64_t u, uint64_t ids, uint64_t stream) {
    clear_error();
    if (!s) return fail("sz_head_argmax: null session");
    return head_argmax(s, m, u, ids, stream);
}

int32_t sz_head_logits(sz_session* s, uint32_t m, uint64_t u, uint64_t logits, uint64_t stream) {
    clear_error();
    if (!s) return fail("sz_head_logits: null session");
    return head_logits(s, m, u, logits, stream);
}

// The merge kernel's output goes straight into pinned host memory (device-visible, coherent): once the stream has drained the
// 512 bytes a row are there, and no copy from device memory (a blocking driver call of its own) is needed.
static int top_finish(sz_session* s, uint32_t m, uint32_t* top_host, uint64_t stream) {
    if (sz_stream_synchronize(stream)) return 1;
    std::memcpy(top_host, s->top_host, (size_t) m * 128 * 4);
    return 0;
}

int32_t sz_head_top(sz_session* s, uint32_t m, uint64_t u, uint32_t* top_host, uint64_t stream) {
    clear_error();
    if (!s) return fail("sz_head_top: null session");
    if (!s->top_host && hip_check(hip().hipHostMalloc(&s->top_host, 8 * 128 * 4, 0), "hipHostMalloc")) return 1;
    const uint64_t topo = (uint64_t) s->top_host;
    const sz_session_config& c = s->cfg;
    const uint32_t nb = (c.vocab + 4095) / 4096;
    if (nb > 64) return fail("sz_head_top: vocabulary above 262144");
    if (head_check(s, m, u, "sz_head_top")) return 1;
    if (s->hp.k_blk) {   // head_top_at, session.rs:5997-6022: the screened form, the top 64 among the chosen blocks
        if (s->topv.need(8ull * 64 * 64 * 4) || s->topi.need(8ull * 64 * 64 * 4)) return 1;
        uint32_t max_sel = 0;
        if (head_proxy_sparse(s, m, u, 64, &max_sel, stream)) return 1;
        const uint32_t nbs = (max_sel * 128 + 4095) / 4096;
        const sz_arg a[] = {P(s->hp.logits.ptr), U32(max_sel * 128), P(s->hp.sel.ptr), U32(nbs), P(s->topv.ptr), P(s->topi.ptr)};
        if (launch("topk_slices_blks", m * nbs, 1, 1, 1024, 0, stream, a)) return 1;
        const sz_arg b[] = {P(s->topv.ptr), P(s->topi.ptr), U32(nbs), P(topo)};
        if (launch("topk_merge", m, 1, 1, 1024, 0, stream, b)) return 1;
        return top_finish(s, m, top_host, stream);
    }
    if (s->logits.need((uint64_t) c.max_rows * c.vocab * 4)) return 1;
    if (head_logits(s, m, u, s->logits.ptr, stream)) return 1;
    if (head_is_exl3(s)) {   // its blocks' largest logits say which blocks hold the 64
        const sz_arg a[] = {P(s->logits.ptr), U32(c.vocab), P(s->head_part.ptr), U32(c.vocab / 128), P(topo)};
        if (launch("topk_blocks", m, 1, 1, 1024, 0, stream, a)) return 1;
        return top_finish(s, m, top_host, stream);
    }
    if (s->topv.need((uint64_t) c.max_rows * nb * 64 * 4) || s->topi.need((uint64_t) c.max_rows * nb * 64 * 4)) return 1;
    const sz_arg a[] = {P(s->logits.ptr), U32(c.vocab), U32(c.vocab), U32(nb), P(s->topv.ptr), P(s->topi.ptr)};
    if (launch("topk_slices", m * nb, 1, 1, 1024, 0, stream, a)) return 1;
    const sz_arg b[] = {P(s->topv.ptr), P(s->topi.ptr), U32(nb), P(topo)};
    if (launch("topk_merge", m, 1, 1, 1024, 0, stream, b)) return 1;
    return top_finish(s, m, top_host, stream);
}

int32_t sz_verify_accept(const uint32_t* ids, const uint32_t* drafts, uint32_t n_drafts, uint32_t* keep) {
    clear_error();
    uint32_t k = 1;
    for (uint32_t i = 0; i < n_drafts; i++) {
        if (ids[i] != drafts[i]) break;
        k++;
    }
    *keep = k;
    return 0;
}

int32_t sz_lookup_draft(const uint32_t* hist, uint64_t n_hist, uint32_t k, const uint32_t* lens, uint32_t n_lens, uint32_t* drafts, uint32_t* n_drafts) {
    clear_error();
    if (!n_drafts || (n_hist && !hist) || (n_lens && !lens) || (k && !drafts)) return fail("sz_lookup_draft: null argument");
    *n_drafts = 0;
    for (uint32_t li = 0; li < n_lens; li++) {
        const uint64_t n = lens[li];
        if (k == 0 || n_hist <= n) break;   // as the reference: a length the history cannot hold ends the search
        const uint32_t* tail = hist + n_hist - n;
        for (uint64_t i = n_hist - n; i-- > 0;) {   // the most recent earlier occurrence first
            if (std::memcmp(hist + i, tail, n * 4) != 0) continue;
            const uint64_t end = std::min<uint64_t>(i + n + k, n_hist);
            for (uint64_t j = i + n; j < end; j++) drafts[(*n_drafts)++] = hist[j];
            return 0;
        }
    }
    return 0;
}

int32_t sz_verify_round(sz_session* s, uint32_t m, uint64_t u, uint64_t rl, uint64_t sgl, uint64_t y, uint64_t head_u, uint64_t drafts,
                        uint64_t out, uint64_t stream) {
    clear_error();
    if (!s) return fail("sz_verify_round: null session");
    if (m == 0 || m > s->cfg.max_rows) return fail("sz_verify_round: " + std::to_string(m) + " rows");
    const sz_session_config& c = s->cfg;
    // everything that can be refused is refused before a capture begins
    if (head_check(s, m, head_u, "sz_verify_round")) return 1;
    if ((u & 15) || (y & 15)) return fail("sz_verify_round: activations must be 16-byte aligned");
    for (uint32_t l = 0; l < c.n_layers; l++) {
        const SzLayer& L = s->layers[l];
        if (!L.set) return fail("sz_verify_round: layer " + std::to_string(l) + " has no experts set");
        if (L.shared && L.shared_type != L.type) return fail("the shared expert must have the routed experts' type (layer " + std::to_string(l) + ")");
    }
    const SzGraphKey key{{m, u, rl, sgl, y, head_u, drafts, out, stream, 0}};
    auto it = s->use_graph ? s->graphs.find(key) : s->graphs.end();
    if (it == s->graphs.end()) {
        static const bool no_graph = std::getenv("SHADOWZERO_NO_GRAPH") != nullptr;
        auto record = [&]() -> int {
            // every layer's inputs are given: the EXL3 layers go through the verify launches together, whatever their order
            if (!s->vtab.empty() && verify_layers(s, 0, (uint32_t) s->vtab.size(), 0, m, u, rl, sgl, y, s->plans.ptr, stream)) return 1;
            for (uint32_t l = 0; l < c.n_layers; l++) {
                if (s->layers[l].type > 1020) {
                    s->last_plan = s->plans.ptr + (uint64_t) l * s->plan_stride;
                    s->last_fused = true;
                    continue;
                }
                const uint64_t off = (uint64_t) l * m;
                if (moe_layer(s, l, m, u + off * c.hidden * 4, rl + off * c.n_expert * 4, sgl + off * 4, y + off * c.hidden * 4, stream)) return 1;
            }
            const Accept acc{drafts, out};
            return head_argmax(s, m, head_u, out + 8, stream, &acc);
        };
        if (no_graph || !s->use_graph || stream == 0) return record();   // the null stream cannot be captured
        if (sz_capture_begin(stream)) return 1;
        const int r = record();
        const std::string err = r ? sz_last_error() : "";
        uint64_t exec = 0;
        const int e = sz_capture_end(stream, &exec);
        if (r) {
            if (!e && exec) sz_graph_destroy(exec);   // a graph of a round that could not be recorded is not kept
            return fail(err);
        }
        if (e) return 1;
        it = s->graphs.emplace(key, SzRoundGraph{exec, s->last_plan, s->last_fused}).first;
    }
    s->last_plan = it->second.plan;
    s->last_fused = it->second.fused;
    return sz_graph_launch(it->second.exec, stream);
}

int32_t sz_quantize_act(uint64_t x, uint64_t n, uint64_t q, uint64_t d, uint64_t stream) {
    clear_error();
    if (n % 32) return fail("sz_quantize_act: the length must be a multiple of 32");
    if (n == 0) return 0;
    const sz_arg a[] = {P(x), U64(n), P(q), P(d)};
    return launch("quant_act_q8", (uint32_t) ((n / 32 + 255) / 256), 1, 1, 256, 0, stream, a);
}

int32_t sz_moe_prefill_chunk(sz_session* s, uint32_t l, uint32_t tokens, uint64_t x, uint64_t rl, uint64_t sgl, uint64_t y, uint64_t stream) {
    clear_error();
    if (!s) return fail("sz_moe_prefill_chunk: null session");
    const sz_session_config& c = s->cfg;
    if (l >= s->layers.size() || !s->layers[l].set) return fail("sz_moe_prefill_chunk: layer " + std::to_string(l) + " has no experts set");
    SzLayer& L = s->layers[l];
    Format f;
    std::string tag;
    format_of(L.type, f, tag);
    const bool exl3 = f.exl3 && !f.half;
    if ((L.type != SZ_TYPE_IQ3_S && !exl3) || (L.shared && L.shared_type != L.type))
        return fail("sz_moe_prefill_chunk: the chunk kernels are built for IQ3_S experts (int8 activations) and EXL3 experts at a whole bit rate");
    if (tokens == 0 || tokens > 16384) return fail("sz_moe_prefill_chunk: " + std::to_string(tokens) + " tokens (1..16384)");   // BIG_BATCH_MAX, session.rs:191
    if (c.hidden % 256 || c.ff % 256 || (x & 15) || (y & 15)) return fail("sz_moe_prefill_chunk: shapes must be multiples of 256 and 16-byte aligned");
    const bool shared = L.shared != 0;
    const uint64_t T = tokens, k = c.top_k, np = T * k, rows = np + (shared ? T : 0);
    auto& pb = s->pf;
    // prefill_group: one workgroup up to 4096 pairs, beyond them one for the items and up to 16 that list 2048 pairs or more each
    auto group = [&](uint64_t items_d, uint32_t unit, uint32_t unit_d) -> int {
        const sz_arg a[] = {P(pb.tidx.ptr), U32(tokens), U32(c.top_k), U32(c.n_expert), U32(shared ? tokens : 0), P(pb.offs.ptr), P(pb.list.ptr), P(pb.items.ptr), P(items_d), U32(unit), U32(unit_d)};
        if (np <= 4096) return launch("prefill_group", 1, 1, 1, 1024, 0, stream, a);
        const uint32_t share = (uint32_t) std::max<uint64_t>(2048, (np + 15) / 16);
        const sz_arg b[] = {a[0], a[1], a[2], a[3], a[4], a[5], a[6], a[7], a[8], a[9], a[10], U32(share)};
        return launch("prefill_group_many", 1 + (uint32_t) ((np + share - 1) / share), 1, 1, 1024, 0, stream, b);
    };
    if (exl3) {
        // EXL3 experts: f16 activations on the columns of the matrix instruction, items of up to 128 pairs, of 64 for the down
        // products (kernels/exl3.hip, "the prefill chunk of an EXL3 layer": XPF_NT, XPF_DOWN_NT, XPF_ROWS_U16, XPF_RING)
        if (c.ff > 512) return fail("sz_moe_prefill_chunk: EXL3 experts of more than 512 intermediate features are not built (a workgroup keeps four 128-blocks of a token)");
        const uint32_t kbs = c.hidden / 128, fbs = c.ff / 128;
        const uint64_t some = std::min<uint64_t>(c.n_expert, np) + 1;
        // The gate and up launch: workgroups of one 128-block of ff, two of which share a compute unit, with items of up to 64 pairs; for long
        // chunks of two 128-blocks and items of up to 128 pairs: an expert is decoded less often, but a workgroup has a unit for
        // itself (4096 tokens through 512 experts of 2048 x 512, top-10, and the shared one, 4 bits, one block and two, a router with
        // Zipf's preferences: 941 and 915 us, without: 1110 and 1019; 3500 through 64 of 3072 x 512, top-6: 727 and 681; 2048 as the first
        // 556 and 550, 601 and 669; 4000 through 256 of 3072 x 256, top-6, 2 bits 611 and 624; measured again since both gained: 1500 as the
        // first 433, 433, 512 of them 221, 218, 200 140, 172).
        const bool wide_gu = rows * fbs >= 95000;
        // Of one block, items so short that the chip is full: an item's chain over all inputs takes about 4 + its tiles; two workgroups that share
        // a unit 1.6 times that.  Routers prefer some experts: 0.3 of those that independent choices would reach, the experts' last tiles
        // and the rest of the pairs in whole items.  us with items of 16, 32 and 64 pairs, router with Zipf's preferences and without: 45 tokens
        // as above at 3 bits 100, 112, 106 and 213, 240, 240; 200 tokens 179, 160, 140 and 354, 335, 347; 512 tokens 328, 260, 227 and
        // 384, 395, 395; 200 through 128 of 4096 x 512, top-8, and the shared one, 4 bits 244, 196, 206 and 243, 244, 246; 300 through 160
        // of 2560 x 256, top-6, 121, 105, 132 and 123, 127, 141; 500 through 32 of 2048 x 512, top-2, 3 bits 101, 82, 99.
        const double reached = 0.3 * c.n_expert * (1.0 - std::pow(1.0 - (double) c.top_k / c.n_expert, (double) T));
        uint32_t most = f.bits <= 5 ? 8 : 6;   // XPF_NT
        if (!wide_gu) {
            double best = 1e30;
            for (uint32_t n : {4u, 2u, 1u}) {
                const double chain = 4 + (double) std::min<uint64_t>(n, (T + 15) / 16), rest = (double) rows / (16 * n);
                const double cost = (reached + rest) * fbs <= 256 ? chain : std::max(1.6 * chain, 0.95 / 256 * fbs * (reached * 5 + rest * chain));
                if (cost < best) best = cost, most = n;
            }
        }
        const uint32_t tok = 16 * most, ntl = std::min<uint32_t>(most, (tokens + 15) / 16), nt = ntl <= 2 ? ntl : ntl + ntl % 2, nd = std::min(4u, nt);
        const uint64_t max_items = some + rows / tok, max_down = some + rows / (16 * nd), tiles = rows / 16 + c.n_expert + 2;
        // (room for items of one tile whatever their length: a chunk never takes more than a longer one)
        const uint32_t bound = (uint32_t) ((max_items + 7) / 8 * 8), bound_d = (uint32_t) ((max_down + 7) / 8 * 8);   // workgroups an item's part (xpf_place)
        if (pb.lay({{&pb.tidx, np * 4}, {&pb.w, np * 4}, {&pb.cnt, T * 4}, {&pb.offs, (c.n_expert + 2) * 4ull}, {&pb.list, rows * 4}, {&pb.items, (2 + 4 * (some + rows / 16)) * 4},
                    {&pb.eo, rows * c.hidden * 4}, {&pb.most, T * 8}, {&pb.arows, tiles * 2 * kbs * 4096}, {&pb.ainv, tiles * 2 * 64}, {&pb.drows, tiles * fbs * 4096}, {&pb.dinv, tiles * fbs * 64}}))
            return 1;
        const uint64_t sh = shared ? L.eaddr.ptr + 3ull * c.n_expert * 8 : 0, items_d = pb.items.ptr + (1 + 2 * max_items) * 4;
        {
            const sz_arg a[] = {P(rl), P(pb.tidx.ptr), P(pb.w.ptr), P(pb.cnt.ptr), U32(c.n_expert), U32(c.top_k), U32(tokens), P(x), P(pb.most.ptr), U32(c.hidden)};
            if (launch("route_topk_rows", (tokens + 3) / 4 * 2, 1, 1, 256, 0, stream, a)) return 1;
        }
        if (group(items_d, tok, 16 * nd)) return 1;
        {
            // shares of the inputs' 128-blocks, as many as make about 1200 workgroups of a few tiles (45 tokens through 512 experts of 2048 x 512
            // as above 121, 118, 117, 115 us with 1 to 4, 250 as above 159, 152, 146, 150, 1200 through 128 of 4096 x 512, top-8, at 4 bits
            // 574, 564, 563, 561)
            const uint32_t shares = (uint32_t) std::max(1.0, std::min<double>(kbs / 4, std::floor(1200.0 / (reached + rows / 16) + 0.5)));
            const sz_arg a[] = {P(L.eaddr.ptr), P(sh), P(pb.offs.ptr), P(pb.list.ptr), P(pb.items.ptr), P(x), P(pb.most.ptr), P(pb.arows.ptr), P(pb.ainv.ptr), U32(c.n_expert),
                                U32(c.top_k), U32((uint32_t) np), U32(c.hidden), U32(tok), U32(ntl), U32(shares)};
            if (launch("prefill_rotate_exl3", bound * ntl * shares, 1, 1, 256, 0, stream, a)) return 1;
        }
        const uint32_t bits = (uint32_t) f.bits, wide_ring = bits <= 7 ? 3 : 2;
        {
            const uint32_t ncb = wide_gu ? 2 : 1;
            // LDS: slots of a unit's operand rows and the rings of trellis rows (XPF_RING_W, XPF_RING_N), afterwards the exchange of four tiles' sums
            uint32_t lds = ncb * 2 * std::min(4u, nt) * 8192;
            for (uint32_t n = 1; n <= nt; n += n == 1 ? 1 : 2) {
                const uint32_t ring = !wide_gu ? std::min(8u, (40 - 2 * n) / (2 * n + bits)) : n >= 6 ? wide_ring : std::min(8u, (39 - n) / (n + bits));
                lds = std::max(lds, (wide_gu && n >= 6 ? 3 : ring + 1) * 2 * n * 2048 + 4 * ncb * ring * 512 * bits);
            }
            const sz_arg a[] = {P(L.eaddr.ptr), P(sh), P(pb.offs.ptr), P(pb.items.ptr), P(pb.arows.ptr), P(pb.ainv.ptr), P(pb.drows.ptr), P(pb.dinv.ptr), U32(c.n_expert), U32(c.hidden), U32(c.ff), U32(tok)};
            if (launch(((wide_gu ? "prefill_gate_up_" : "prefill_gate_up_n_") + tag).c_str(), bound * (fbs / ncb), 1, 1, 512, lds, stream, a)) return 1;
        }
        {
            // shares of an item: a wave a column block, but all blocks on eight waves, whose start then counts once, where items fill the chip (1, 2
            // shares of 8 waves, 4 of 4: 45 tokens as above 137, 109, 101 us, 512 tokens 257, 252, 267, 4096 at 4 bits 967, 988, 1071; 4 and
            // 8 shares of 4: 64 tokens through 60 of 4096 x 512, top-4, 4 bits 167, 150; 8 and 4 waves: 764 tokens, top-3 of 128 of 1792 x 256
            // and the shared one, 2 bits 142, 132, 700 through 64 of 1024 x 256, top-4, 97, 93, 380 through 256 of 3072 x 256, top-8, at 5
            // bits 230, 242, 190 as above 178, 182)
            const bool wide = rows * fbs * kbs >= 115000;
            const uint32_t waves = std::min(wide ? 8u : 4u, kbs), parts = rows >= 20000 ? (kbs + 4 * waves - 1) / (4 * waves) : (kbs + waves - 1) / waves;
            const uint32_t ring = wide ? wide_ring : bits <= 3 ? 8 : bits == 4 ? 7 : bits == 5 ? 5 : bits <= 7 ? 4 : 3;   // XPF_RING, XPF_RING_DOWN_N
            const sz_arg a[] = {P(L.eaddr.ptr), P(sh), P(pb.offs.ptr), P(pb.list.ptr), P(items_d), P(pb.drows.ptr), P(pb.dinv.ptr), P(pb.eo.ptr), U32(c.n_expert), U32(c.hidden), U32(c.ff),
                                U32(nd), U32(parts)};
            if (launch(((wide ? "prefill_down_" : "prefill_down_n_") + tag).c_str(), bound_d * parts, 1, 1, 64 * waves, 4 * (nd * fbs * 1040 + 256 * waves) + waves * ring * 512 * bits, stream, a)) return 1;
        }
        const sz_arg a[] = {P(y), P(pb.eo.ptr), P(pb.w.ptr), P(shared ? pb.eo.ptr + np * c.hidden * 4 : 0), P(sgl), P(pb.cnt.ptr), U32(c.hidden / 4), U32(c.top_k)};
        return launch("prefill_combine", c.hidden / 256, tokens, 1, 64, 0, stream, a);
    }
    const uint64_t max_items = c.n_expert + 1 + rows / 64;   // every expert's runs of up to 64 pairs: PF_TOK in kernels/prefill.hip
    if (pb.lay({{&pb.xq, T * c.hidden}, {&pb.xd, T * c.hidden / 32 * 4}, {&pb.tidx, np * 4}, {&pb.w, np * 4}, {&pb.cnt, T * 4}, {&pb.offs, (c.n_expert + 2) * 4ull}, {&pb.list, rows * 4},
                {&pb.items, (1 + 2 * max_items) * 4}, {&pb.hq, rows * c.ff}, {&pb.xh, T * c.hidden * 2}, {&pb.hh, rows * c.ff * 2}, {&pb.hd, rows * (c.ff / 32) * 4}, {&pb.eo, rows * c.hidden * 4}}))
        return 1;
    const uint64_t sh = shared ? L.eaddr.ptr + 3ull * c.n_expert * 8 : 0;
    {
        // routing and quantization do not depend on each other: one launch
        const uint64_t n = T * c.hidden;
        const sz_arg a[] = {P(x), U64(n), P(pb.xq.ptr), P(pb.xd.ptr), P(pb.xh.ptr), P(rl), P(pb.tidx.ptr), P(pb.w.ptr), P(pb.cnt.ptr), U32(c.n_expert), U32(c.top_k), U32(tokens)};
        if (launch("prefill_front", (tokens + 3) / 4 + (uint32_t) ((n / 32 + 255) / 256), 1, 1, 256, 0, stream, a)) return 1;
    }
    if (group(0, 64, 64)) return 1;
    {
        const sz_arg a[] = {P(L.eaddr.ptr), P(sh), P(pb.offs.ptr), P(pb.list.ptr), P(pb.items.ptr), P(pb.xh.ptr), P(pb.xd.ptr), P(pb.hq.ptr), P(pb.hh.ptr), P(pb.hd.ptr),
                            U32(c.n_expert), U32(c.top_k), U32((uint32_t) np), U32(c.hidden), U32(c.ff)};
        if (launch("prefill_gate_up_iq3_s", c.ff / 64, (uint32_t) max_items, 1, 512, 0, stream, a)) return 1;
    }
    {
        // 128 rows a workgroup; in long chunks, which fill the chip many times over, four lots in turn, whose set-up counts once (1, 2 and 4 lots:
        // 4096 tokens through 512 experts of 2048 x 512, top-10, and the shared one 861, 851, 847 us; 512 tokens 174, 174, 178, 150 through
        // 128 of 2560 x 768, top-8, 120, 125, 128, 40 through 64 of 1024 x 256, top-4, 30, 33, 38)
        const uint32_t blocks = c.hidden / 128, per = rows >= 20000 && blocks % 4 == 0 ? 4 : 1;
        const sz_arg a[] = {P(L.eaddr.ptr), P(sh), P(pb.offs.ptr), P(pb.list.ptr), P(pb.items.ptr), P(pb.hh.ptr), P(pb.hd.ptr), P(pb.eo.ptr), U32(c.n_expert),
                            U32(c.hidden), U32(c.ff)};
        if (launch("prefill_down_iq3_s", blocks / per, (uint32_t) max_items, 1, 512, 0, stream, a)) return 1;
    }
    const sz_arg a[] = {P(y), P(pb.eo.ptr), P(pb.w.ptr), P(shared ? pb.eo.ptr + np * c.hidden * 4 : 0), P(sgl), P(pb.cnt.ptr), U32(c.hidden / 4), U32(c.top_k)};
    return launch("prefill_combine", c.hidden / 256, tokens, 1, 64, 0, stream, a);
}

// The chunk's intermediate buffers, for tests: which = 0 xq (int8), 1 xd (f32), 2 tidx (u32), 3 w (f32), 4 hq (int8), 5 hd (f32),
// 6 eo (f32), 7 xh and 8 hh (f16, the codes the products read).  Returns the device address (0 if the session has not run a chunk).
uint64_t sz_prefill_buffer(sz_session* s, int32_t which) {
    if (!s) return 0;
    auto& pb = s->pf;
    const uint64_t ptrs[] = {pb.xq.ptr, pb.xd.ptr, pb.tidx.ptr, pb.w.ptr, pb.hq.ptr, pb.hd.ptr, pb.eo.ptr, pb.xh.ptr, pb.hh.ptr};
    return which >= 0 && which < (int32_t) (sizeof ptrs / sizeof ptrs[0]) ? ptrs[which] : 0;
}

}   // extern "C"

// ---- the hyper-connection around a sublayer ---------------------------------------------------------------------------------
struct sz_hc {
    sz_hc_config cfg{};
    DevBuf scales, down, g;   // f64[max_rows][streams], f32[max_rows][rank], f32[max_rows][streams]
};

extern "C" {

sz_hc* sz_hc_new(const sz_hc_config* cfg) {
    clear_error();
    if (ensure_init()) return nullptr;
    const sz_hc_config& c = *cfg;
    const uint64_t ch = (uint64_t) c.hidden * c.streams;
    Format fd, fu, fi;
    std::string td, tu, ti;
    if (c.hidden == 0 || c.hidden % 4 || c.streams == 0 || c.streams > 64 || c.rank == 0 || c.rank % 4 || c.max_rows == 0 || c.max_rows > 8 || ch >> 31) {
        fail("sz_hc_new: hidden and rank must be multiples of 4, streams 1..64, max_rows 1..8");
        return nullptr;
    }
    if (!format_of(c.down_type, fd, td) || !fd.dense || !format_of(c.up_type, fu, tu) || !fu.dense ||
        (c.inject_w && (!format_of(c.inject_type, fi, ti) || !fi.dense))) {
        fail("sz_hc_new: the projections must be F32, F16 or BF16");
        return nullptr;
    }
    if (!c.norm_w || !c.down_w || !c.up_w || (c.norm_w & 3) || (c.down_w & (4 * fd.bb - 1)) || (c.up_w & (4 * fu.bb - 1)) ||
        (c.inject_w & (4 * (c.inject_w ? fi.bb : 1) - 1))) {
        fail("sz_hc_new: weights must be resident and aligned to four weights");
        return nullptr;
    }
    sz_hc* h = new sz_hc();
    h->cfg = c;
    if (h->scales.need((uint64_t) c.max_rows * c.streams * 8) || h->down.need((uint64_t) c.max_rows * c.rank * 4) || h->g.need((uint64_t) c.max_rows * c.streams * 4)) {
        delete h;
        return nullptr;
    }
    return h;
}

void sz_hc_free(sz_hc* h) { delete h; }
uint64_t sz_hc_gains(sz_hc* h) { return h ? h->g.ptr : 0; }

int32_t sz_hc_read(sz_hc* h, uint32_t m, uint64_t r, uint64_t u, uint64_t stream) {
    clear_error();
    if (!h) return fail("sz_hc_read: null handle");
    const sz_hc_config& c = h->cfg;
    if (m == 0 || m > c.max_rows) return fail("sz_hc_read: " + std::to_string(m) + " rows (1.." + std::to_string(c.max_rows) + ")");
    if ((r & 15) || (u & 15)) return fail("sz_hc_read: rows must be 16-byte aligned");
    const DenseShape d = dense_shape((uint64_t) c.hidden * c.streams);
    const uint32_t group = d.block / 64 / d.waves;   // whole rows, a wave or more each
    const uint64_t ch = (uint64_t) c.hidden * c.streams;
    const uint32_t groups = (c.rank + group - 1) / group + (c.inject_w ? (c.streams + group - 1) / group : 0);
    const DenseShape du = dense_shape(c.rank);
    const uint32_t per = 4 * std::max<uint32_t>(1, du.pass / (du.block / 64 / du.waves));   // 4 waves of 64 / G columns
    // LDS of the first launch: the sums of squares of every stream's spans (of at least 256 columns) and its scale; as many rows
    // at a time as fit half a compute unit's (all of them, unless the streams are many and long)
    const bool eight = c.hidden % 8 == 0 && c.down_type != SZ_TYPE_F32 && (!c.inject_w || c.inject_type != SZ_TYPE_F32);
    const uint64_t lds = (uint64_t) c.streams * (c.hidden / (eight ? 512 : 256) + 3) * 8;
    const uint32_t lot = (uint32_t) std::min<uint64_t>(m, std::max<uint64_t>(1, 80000 / lds));
    for (uint32_t j = 0; j < m; j += lot) {
        const uint32_t n = std::min(lot, m - j);
        // Rows one after the other in a workgroup of the first launch, as many (of its 4) as bring the launch down to a workgroup a
        // compute unit: each normalises all inputs in f64 for itself, and two on one unit take turns at that.  A read and a write,
        // bf16, rank 320: 4 rows of 8192 columns 19.1 us with 324 workgroups of a row, 17.0 with 162 of two (17.4 with three), 4 rows
        // of 16384 28.3 and 24.9; rank 512: 6 rows of 6144 37.7 us with a row each, 24.9 with three.  One row of more than 8192
        // columns, which has little to normalise and is bound by its loads' latency, is better off with two workgroups a unit: 17.6
        // and 18.1 us.  A row each has kernels of its own (the loop over rows costs them 3 to 5%).
        const uint32_t units = n == 1 && ch > 8192 ? 512 : 256, np = std::min(4u, (groups + units - 1) / units), pass = group * np;
        const uint64_t rj = r + (uint64_t) j * c.hidden * c.streams * 4, sc = h->scales.ptr + (uint64_t) j * c.streams * 8, dj = h->down.ptr + (uint64_t) j * c.rank * 4;
        const sz_arg a[] = {U32(dense_code(c.down_type)), P(c.down_w), U32(c.rank), U32(dense_code(c.inject_type)), P(c.inject_w), P(rj), P(c.norm_w), P(sc),
                            P(dj), P(h->g.ptr + (uint64_t) j * c.streams * 4), U32(c.hidden), U32(c.streams), U32(n), F32(c.eps), U32(np)};
        if (launch((std::string(np > 1 ? "hc_down_rows_m" : "hc_down_m") + dense_m(n)).c_str(),
                   (c.rank + pass - 1) / pass + (c.inject_w ? (c.streams + pass - 1) / pass : 0), 1, 1, d.block, (uint32_t) (n * lds), stream, a))
            return 1;
        const sz_arg b[] = {U32(dense_code(c.up_type)), P(c.up_w), P(dj), P(rj), P(c.norm_w), P(sc), P(u + (uint64_t) j * c.hidden * 4), U32(c.hidden), U32(c.streams), U32(c.rank), U32(n)};
        if (launch((std::string("hc_up_m") + dense_m(n)).c_str(), (c.hidden + per - 1) / per, 1, 1, 256, 0, stream, b)) return 1;
    }
    return 0;
}

int32_t sz_hc_write(uint64_t r, uint64_t g, uint64_t y, uint32_t m, uint32_t hidden, uint32_t streams, uint64_t stream) {
    clear_error();
    if (m == 0 || hidden == 0 || streams == 0 || streams > 65535 || m > 65535) return fail("sz_hc_write: bad shape");
    const sz_arg a[] = {P(r), P(g), P(y), U32(hidden), U32(streams)};
    return launch("hc_write_rows", (hidden + 255) / 256, streams, m, 256, 0, stream, a);
}

}   // extern "C"
