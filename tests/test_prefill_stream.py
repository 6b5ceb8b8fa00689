"""The order of requests, waits and reads of the EXL3 prefill chunk's product streams, on the CPU: the streams' own source, compiled for the
host with their loads, waits and LDS reads replaced by checks, in the forms that the gate and up kernel instantiates."""
import os
import re
import subprocess

from shadow_engine_amd import build

HARNESS = r"""
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <map>
typedef uint8_t u8; typedef uint16_t u16; typedef uint32_t u32; typedef uint64_t u64;
typedef float f32x4 __attribute__((vector_size(16)));
typedef u32 u32x4 __attribute__((vector_size(16)));
#define __device__
#define __forceinline__ inline
#define __builtin_amdgcn_readfirstlane(x) (x)
#define __builtin_amdgcn_sched_barrier(x)
#define __builtin_amdgcn_s_waitcnt(x)
%(macros)s

struct Slot { u32 unit; long last; };   // what a slot holds and the number of its last load
static long issued, landed;             // loads made, and how many of them have arrived for certain
static std::map<long, Slot> trellis, operands;
static u32 units, tiles, part, parts, words, slot_halves, step;   // step: which read of the stream comes next
static const u16 *source, *lds_rows;
static const u32* lds_words;
static const char* what;
static void check(bool ok, const char* fault) {
    if (ok) return;
    printf("%%s: units %%u, tiles %%u, wave %%u of %%u, step %%u: %%s\n", what, units, tiles, part, parts, step, fault);
    exit(1);
}
static u32 lds_offset(const void* p) { return (u32) ((const u8*) p - (const u8*) lds_rows); }
template <int B> static void lds_load(const u8* from, u32 to) {
    const long at = from - (const u8*) source;
    check(at >= 0 && at + 1024 <= (long) units * tiles * 2048, "operand rows past the item's");
    const u32 unit = at / (2048 * tiles), slot = to / (2 * slot_halves);
    if (operands.count(slot) && operands[slot].unit != unit) check(2 * operands[slot].unit + 1 < step, "a slot is filled before it was read");
    operands[slot] = {unit, ++issued};
}
template <int N> static void wait_vm() { landed = issued - N > landed ? issued - N : landed; }
static void lds_barrier() {}
template <int DEPTH, int LOADS> struct Ring {
    static constexpr int D = DEPTH, UR = 4, NI = LOADS, UW = 64;
    u32 units;
    void issue(u32 unit, u32 slot, u32) const {
        check(unit < units, "a unit past the stream's end");
        if (trellis.count(slot)) check(2 * trellis[slot].unit + 1 < step, "a ring slot is filled before it was read");
        trellis[slot] = {unit, issued += NI};
    }
};
template <int K, int CT, int NT> struct XpfStep {
    void read(const u32* row, u32 s, u32) {
        const Slot& t = trellis[(row - lds_words) / 64];
        check(t.unit == step / 2 && s == step %% 2, "another unit's words");
        check(t.last <= landed, "words that have not landed");
    }
    static void rows(u32x4 (&)[NT], const u16* xa, u32) {
        if (part < 2 * tiles) {   // this wave's share of them: the others wait for theirs before the barrier
            const Slot& t = operands[(xa - lds_rows) / slot_halves];
            check(t.unit == step / 2, "another unit's operand rows");
            check(t.last <= landed, "operand rows that have not landed");
        }
        step++;
    }
    template <int c0> void products(const u32x4 (&)[NT], f32x4 (&)[NT][CT], u32) const {}
};
%(stream)s

template <int K, int NT, int NCB> static void stream(const char* name) {
    constexpr int CT = NCB == 2 ? 4 : 2, WAVES = 4;                      // column tiles a wave, waves a projection
    typedef Ring<%(depth)s, (4 * CT * 2 * K + 63) / 64> R;               // a tile is 2 K times 16 bytes, a load 64 times
    constexpr int NB = %(slots)s;
    // bytes of LDS: the slots of two projections' operand rows and the waves' rings
    static_assert(NB * 2 * NT * 2048 + 2 * WAVES * R::D * 4 * CT * 32 * K <= (NCB == 2 ? 156 : 80) * 1024, "LDS");
    static u16 src[64 * 8 * 1024], rows[9 * 2 * 8 * 1024];
    static u32 wb[16 * 64];
    for (u32 n : {4u, 8u, 12u, 16u, 64u})
        for (u32 t = NT <= 2 ? NT : NT - 1; t <= (u32) NT; t++)
            for (u32 p = 0; p < (u32) WAVES; p++) {
                issued = landed = 0;
                trellis.clear();
                operands.clear();
                what = name, units = n, tiles = t, part = p, parts = WAVES, step = 0, slot_halves = 2 * NT * XPF_HALF_U16, source = src, lds_rows = rows, lds_words = wb;
                f32x4 acc[NT][CT];
                R ring;
                ring.units = n;
                if constexpr (NCB == 2) %(wide)s(ring, wb, src, rows, slot_halves, t, p, 0u, acc);
                else %(narrow)s(ring, wb, src, rows, slot_halves, t, p, 0u, acc);
                check(step == 2 * n, "the stream ended early");
                check(landed == issued, "loads in flight at the end");
            }
}
template <int K, int NT> static void tiles_of() {
    if constexpr (NCB_ == 2 && NT <= XPF_NT(K)) stream<K, NT, 2>("two blocks");
    if constexpr (NCB_ == 1 && NT <= XPF_NT_N) stream<K, NT, 1>("one block");
}
template <int K> static void rate() { tiles_of<K, 1>(); tiles_of<K, 2>(); tiles_of<K, 4>(); tiles_of<K, 6>(); tiles_of<K, 8>(); }
int main() { rate<1>(); rate<2>(); rate<3>(); rate<4>(); rate<5>(); rate<6>(); rate<7>(); rate<8>(); }
"""


def run_streams(tmp_path, blocks):
    src = open(os.path.join(build.KERNELS, "exl3.hip")).read()
    macros = "\n".join(re.search(r"^#define %s\b.*$" % re.escape(n), src, re.M).group(0) for n in ("XPF_NT", "XPF_NT_N", "XPF_RING", "XPF_RING_W", "XPF_RING_N", "XPF_HALF_U16"))
    kernel = src[src.index("void prefill_gate_up_exl3_kernel("):]

    def of_kernel(pattern):
        return re.search(pattern, kernel[:kernel.index("\n}\n")]).group(1)

    def function(head):
        start = src.index(head)
        return src[start:src.index("\n}\n", start) + 3]

    fills = {"macros": f"#define NCB_ {blocks}\n" + macros, "stream": function("template <int K, int NT, int NB, int NW, class R>") + function("template <int K, int NT, int NB, class R>"),
             "depth": of_kernel(r"typedef VerifyRing<K, false, CT, (.*), 4 \* CT, false> R;"), "slots": of_kernel(r"constexpr int NB = (.*);"),
             "wide": of_kernel(r"if constexpr \(NCB == 2\) (xpf_stream<.*>)\(ring"), "narrow": of_kernel(r"else (xpf_stream_n<.*>)\(ring")}
    assert of_kernel(r"constexpr int CT = (.*);") == "NCB == 2 ? 4 : 2"
    path = tmp_path / "stream.cpp"
    path.write_text(HARNESS % fills)
    subprocess.run(["g++", "-std=c++17", "-O1", "-w", "-o", tmp_path / "stream", path], check=True)
    r = subprocess.run([tmp_path / "stream"], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout


def test_prefill_streams_stay_inside_their_item_and_wait_for_what_they_read(tmp_path):
    """Every bit rate and number of token tiles of the workgroups of two 128-blocks, from the shortest stream (hidden = 256: shorter than most
    rings) on: no request past the stream's end, no slot filled before it was read, no read before it has landed, and rings that a compute unit's
    LDS has room for."""
    run_streams(tmp_path, 2)


def test_prefill_streams_of_eight_waves_as_deep_as_their_tiles_leave_room(tmp_path):
    """The rings of up to four tiles: the fewer the tiles the deeper, at most 8 units, and one unit more would not fit."""
    src = open(os.path.join(build.KERNELS, "exl3.hip")).read()
    macros = "\n".join(re.search(r"^#define %s\b.*$" % n, src, re.M).group(0) for n in ("XPF_RING", "XPF_RING_W", "XPF_RING_N"))
    path = tmp_path / "rings.cpp"
    path.write_text("#include <cstdio>\n" + macros + "\nint main() { for (int k = 1; k <= 8; k++) for (int nt = 1; nt <= 4; nt *= 2) printf(\"%d %d %d %d\\n\", k, nt, XPF_RING_W(k, nt), XPF_RING_N(k, nt)); }\n")
    subprocess.run(["g++", "-o", tmp_path / "rings", path], check=True)
    rings = {tuple(map(int, line.split()[:2])): tuple(map(int, line.split()[2:])) for line in subprocess.run([tmp_path / "rings"], capture_output=True, text=True).stdout.splitlines()}
    for (k, nt), (two, one) in rings.items():
        assert 2 <= two <= 8 and 2 <= one <= 8
        assert two == 8 or (two + 2) * 4096 * nt + 4096 * k * (two + 1) > 156 * 1024
        assert one == 8 or (one + 2) * 4096 * nt + 2048 * k * (one + 1) > 80 * 1024
        assert nt == 4 or (two >= rings[k, 2 * nt][0] and one >= rings[k, 2 * nt][1])


def test_prefill_streams_of_narrow_waves(tmp_path):
    """The same for the workgroups of one 128-block, whose waves take 32 columns, four to a projection, and two of which share a unit."""
    run_streams(tmp_path, 1)
