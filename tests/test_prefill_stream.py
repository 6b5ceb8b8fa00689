"""The order of requests, waits and reads of the EXL3 prefill chunk's product streams, on the CPU: xpf_stream's own source, compiled for the
host with its loads, waits and LDS reads replaced by checks."""
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

template <int K, int NT, int NB, int NW, int D> static void stream(const char* name) {
    typedef Ring<D, (2 * K + 3) / 4> R;
    static u16 src[64 * 8 * 1024], rows[9 * 2 * 8 * 1024];
    static u32 wb[16 * 64];
    for (u32 n : {4u, 8u, 12u, 16u, 64u})
        for (u32 t = NT <= 2 ? NT : NT - 1; t <= (u32) NT; t++)
            for (u32 p = 0; p < (u32) NW; p++) {
                issued = landed = 0;
                trellis.clear();
                operands.clear();
                what = name, units = n, tiles = t, part = p, parts = NW, step = 0, slot_halves = 2 * NT * XPF_HALF_U16, source = src, lds_rows = rows, lds_words = wb;
                f32x4 acc[NT][4];
                R ring;
                ring.units = n;
                xpf_stream<K, NT, NB, NW>(ring, wb, src, rows, slot_halves, t, p, 0u, acc);
                check(step == 2 * n, "the stream ended early");
                check(landed == issued, "loads in flight at the end");
            }
}
template <int K, int NT> static void both() {
    if constexpr (NT <= XPF_NT(K)) {
        stream<K, NT, 3, 4, XPF_RING(K)>("eight waves");
        if constexpr (NT <= XPF_NT_N) stream<K, NT, XPF_RING_N(K, NT) + 1, 2, XPF_RING_N(K, NT)>("four waves");
    }
}
template <int K> static void rate() { both<K, 1>(); both<K, 2>(); both<K, 4>(); both<K, 6>(); both<K, 8>(); }
int main() { rate<1>(); rate<2>(); rate<3>(); rate<4>(); rate<5>(); rate<6>(); rate<7>(); rate<8>(); }
"""


def test_prefill_streams_stay_inside_their_item_and_wait_for_what_they_read(tmp_path):
    """Every bit rate, number of token tiles and shape of the gate and up launch, from the shortest stream (hidden = 256: shorter than the
    ring of four waves) on: no request past the stream's end, no slot filled before it was read, no read before it has landed."""
    src = open(os.path.join(build.KERNELS, "exl3.hip")).read()
    macros = "\n".join(re.search(r"^#define %s\b.*$" % re.escape(n), src, re.M).group(0) for n in ("XPF_NT", "XPF_NT_N", "XPF_RING", "XPF_RING_N", "XPF_HALF_U16"))
    start = src.index("template <int K, int NT, int NB, int NW, class R>")
    stream = src[start:src.index("\n}\n", start) + 3]
    path = tmp_path / "stream.cpp"
    path.write_text(HARNESS % {"macros": macros, "stream": stream})
    subprocess.run(["g++", "-std=c++17", "-O1", "-w", "-o", tmp_path / "stream", path], check=True)
    r = subprocess.run([tmp_path / "stream"], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout


def test_prefill_streams_of_eight_waves_as_deep_as_their_tiles_leave_room(tmp_path):
    """The same for the rings of workgroups of eight waves: the fewer the tiles the deeper, and within a compute unit's LDS."""
    src = open(os.path.join(build.KERNELS, "exl3.hip")).read()
    macros = "\n".join(re.search(r"^#define %s\b.*$" % re.escape(n), src, re.M).group(0) for n in ("XPF_NT", "XPF_NT_N", "XPF_RING", "XPF_RING_W", "XPF_RING_N", "XPF_HALF_U16"))
    start = src.index("template <int K, int NT, int NB, int NW, class R>")
    stream = src[start:src.index("\n}\n", start) + 3]
    of_four, of_eight = "stream<K, NT, 3, 4, XPF_RING(K)>", "stream<K, NT, NT >= 6 ? 3 : XPF_RING_W(K, NT) + 1, 4, XPF_RING_W(K, NT)>"
    room = "static_assert((NT >= 6 ? 3 : XPF_RING_W(K, NT) + 1) * NT + K * XPF_RING_W(K, NT) <= 39, \"LDS\"); "
    assert of_four in HARNESS
    path = tmp_path / "stream.cpp"
    path.write_text(HARNESS.replace(of_four, room + of_eight) % {"macros": macros, "stream": stream})
    subprocess.run(["g++", "-std=c++17", "-O1", "-w", "-o", tmp_path / "stream", path], check=True)
    r = subprocess.run([tmp_path / "stream"], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout


def test_prefill_streams_of_narrow_waves(tmp_path):
    """The same for the workgroups of one 128-block, whose waves take 32 columns, four to a projection."""
    src = open(os.path.join(build.KERNELS, "exl3.hip")).read()
    macros = "\n".join(re.search(r"^#define %s\b.*$" % re.escape(n), src, re.M).group(0) for n in ("XPF_NT", "XPF_NT_N", "XPF_RING", "XPF_RING_N", "XPF_HALF_U16"))
    start = src.index("template <int K, int NT, int NB, class R>")
    stream = src[start:src.index("\n}\n", start) + 3]
    harness = HARNESS.replace("xpf_stream<K, NT, NB, NW>(", "xpf_stream_n<K, NT, NB>(").replace("f32x4 acc[NT][4];", "f32x4 acc[NT][2];").replace("Ring<D, (2 * K + 3) / 4> R;", "Ring<D, (K + 3) / 4> R;")
    harness = harness.replace("stream<K, NT, 3, 4, XPF_RING(K)>(\"eight waves\");", "").replace("XPF_RING_N(K, NT) + 1, 2, XPF_RING_N(K, NT)", "XPF_RING_N(K, NT) + 1, 4, XPF_RING_N(K, NT)")
    assert harness.count("xpf_stream_n<") == 1 and harness.count("eight waves") == 0 and "+ 1, 4, XPF_RING_N" in harness
    path = tmp_path / "stream.cpp"
    path.write_text(harness % {"macros": macros, "stream": stream})
    subprocess.run(["g++", "-std=c++17", "-O1", "-w", "-o", tmp_path / "stream", path], check=True)
    r = subprocess.run([tmp_path / "stream"], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout
