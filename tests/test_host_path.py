"""The library's host side without a GPU: which launches a call makes, with which addresses, and what a failure leaves behind.
The library binds its HIP runtime at run time, so a child process binds hip_stub.cpp instead, which runs nothing and reports
every launch."""
import os
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)

PRELUDE = '''
import ctypes as C, os
import numpy as np
import shadow_engine_amd as sz
from shadow_engine_amd import synth
stub = C.CDLL(os.environ["SHADOWZERO_HIP_LIB"])
stub.stub_fail_allocations_over.argtypes = [C.c_size_t]
stub.stub_fail_copy_after.argtypes = [C.c_long]
sz.init(0)
PARAMS = {n: k for n, _, k in sz.kernels()}   # kinds: 0, 1 pointers, 2 u32, 3 i32, 4 u64, 5 f32
launches = []
@C.CFUNCTYPE(None, C.c_char_p, C.POINTER(C.c_uint), C.POINTER(C.c_void_p))
def on_launch(name, shape, params):
    name = name.decode()
    ty = {0: C.c_uint64, 1: C.c_uint64, 2: C.c_uint32, 3: C.c_int32, 4: C.c_uint64, 5: C.c_float}
    launches.append((name, tuple(shape[:7]), [ty[k].from_address(params[i]).value for i, k in enumerate(PARAMS[name])]))
stub.stub_on_launch(on_launch)
def taken():
    out = list(launches)
    launches.clear()
    return out
def address(n):   # host memory with room to look like a device buffer
    keep.append(np.zeros(n + 256, np.uint8))
    return (keep[-1].ctypes.data + 255) // 256 * 256
keep = []
'''


@pytest.fixture(scope="module")
def stub(tmp_path_factory):
    so = tmp_path_factory.mktemp("stub") / "libhipstub.so"
    subprocess.run(["g++", "-O1", "-fPIC", "-shared", "-o", str(so), os.path.join(HERE, "hip_stub.cpp")], check=True)

    def run(body):
        env = dict(os.environ, SHADOWZERO_HIP_LIB=str(so), PYTHONPATH=ROOT)
        r = subprocess.run([sys.executable, "-c", PRELUDE + body], env=env, capture_output=True, text=True, timeout=300)
        assert r.returncode == 0, r.stdout + r.stderr
    return run


MIXED = '''
class Layer(C.Structure):
    _fields_ = [("experts", C.c_uint64), ("stride", C.c_uint64), ("shared", C.c_uint64), ("part", C.c_uint32), ("layer", C.c_uint32)]
H, FF, NE, K, M, L, V = 512, 256, 32, 4, 3, 4, 1024
def seen_by(name, shape, a):
    """The layers one of an EXL3 layer's launches works on, as (experts, logits or gate logits, inputs or outputs, plan) each."""
    out = []
    per = {"verify_plan_exl3": 1, "verify_combine_exl3": 1}.get(name, (H + 511) // 512 if "gate_up" in name else (FF + 511) // 512)
    if name == "verify_plan_exl3":
        rl, plans, ps, ioff, table, shared, base = a[:7]
        first, second, e = rl, None, None
    elif name == "verify_combine_exl3":
        dn, table, e, stride, shared, part, base, plans, ps, first, second = a[:11]
    else:
        rl, table, e, stride, shared, part, base, plans, weights, ps, ioff, second = a[:12]
        assert weights == plans
        first = rl
    n = shape[0] if name == "verify_plan_exl3" else shape[2] // per
    for i in range(n):
        lay = Layer.from_address(table + 32 * i) if table else Layer(e or 0, 0, 0, 0, base)
        l = lay.layer - base
        wide = 1 if name == "verify_combine_exl3" else NE
        # without a plan (ioff 0) the ids and weights go to the very place that is given
        assert "combine" in name or ioff or l == 0
        out.append((lay.experts or None, first + l * M * wide * 4, None if "down" in name or second is None else second + l * M * H * 4, plans + l * ps))
    return out
def check(exl3):
    s = sz.Session(H, FF, NE, K, L, V, 8)
    buf = address(1 << 20)                       # nothing reads it
    base = {l: buf + 4096 * l for l in range(L)}
    for l in range(L):
        ty = sz.EXL3(2 + l % 2) if l in exl3 else sz.Q8_0
        s.set_layer(l, ty, base[l], 1 << 20, ty, base[l] + 64)
    s.set_head(sz.Q8_0, address(1024))
    u, rl, sgl, y, hu, dr, out = (address(1 << 16) for _ in range(7))
    taken()
    for replay in range(2):
        s.verify_round(M, u, rl, sgl, y, hu, dr, out, 16)
        got = taken()
        if replay:
            assert not got                       # a graph's replay
            break
        plans = {}
        for name in ("verify_plan_exl3", "verify_gate_up_", "verify_down_", "verify_combine_exl3"):
            done = [x for g in got if g[0].startswith(name) and "q8_0" not in g[0] for x in seen_by(*g)]
            if name == "verify_plan_exl3" and len(exl3) == 1:
                continue                         # a lone layer may do without
            per_layer = {}
            for experts, first, second, plan in done:
                at = (first - (sgl if "combine" in name else rl)) // (M * (1 if "combine" in name else NE) * 4)
                assert at not in per_layer
                per_layer[at] = plan
                assert experts in (None, base[at])
                if second is not None:
                    assert second == (y if "combine" in name else u) + at * M * H * 4
                assert plans.setdefault(at, plan) == plan
            assert sorted(per_layer) == sorted(exl3), (name, per_layer, exl3)
        assert len(set(plans.values())) == len(exl3)
        if L - 1 in exl3:
            assert sz.lib().sz_session_buffer(s._h, 0) == plans[L - 1]
    return s, plans, (u, rl, sgl, y, hu, dr, out)
'''


@pytest.mark.parametrize("exl3", [[0], [1], [3], [1, 2], [0, 3], [0, 1, 2, 3]])
def test_a_round_over_mixed_formats_gives_every_exl3_layer_its_own_buffers(stub, exl3):
    """A round's launches for its EXL3 layers read and write these layers' inputs, plans and outputs, wherever the layers lie among
    GGUF ones and however many there are."""
    stub(MIXED + f"check({exl3})\n")


def test_the_last_routing_after_a_replayed_round_is_the_rounds(stub):
    """Between a round's capture and its replay a single layer's call leaves its own routing; after the replay the last routing is
    the round's last layer's again."""
    stub(MIXED + '''
s, plans, bufs = check([0, 1, 2, 3])
u, rl, sgl, y = bufs[:4]
s.moe_layer_verify(0, M, u, rl, sgl, y, 16)
assert sz.lib().sz_session_buffer(s._h, 0) != plans[L - 1]
taken()
s.verify_round(M, *bufs, 16)
assert not taken() and sz.lib().sz_session_buffer(s._h, 0) == plans[L - 1]
''')


def test_a_layer_that_could_not_be_set_is_not_used(stub):
    """A failed allocation leaves a layer as it was, a failed copy leaves it unset; both are refused by the calls that would run it,
    and setting the layer again mends it."""
    stub(MIXED + '''
s = sz.Session(H, FF, NE, K, L, V, 8)
buf = address(1 << 20)
s.set_head(sz.Q8_0, address(1024))
u, rl, sgl, y, hu, dr, out = (address(1 << 16) for _ in range(7))
def fails(what, f):
    try:
        f()
    except sz.SzError as e:
        assert what in str(e), e
    else:
        raise AssertionError("not refused")
set_layer = lambda l, ty: s.set_layer(l, ty, buf + 4096 * l, 1 << 20, ty, buf + 64)
layer = lambda l: s.moe_layer_verify(l, M, u, rl, sgl, y, 16)
def launched(l, kind):
    taken()
    layer(l)
    got = taken()
    assert got and all(kind in g[0] or g[0].startswith("moe_combine") or g[0].startswith("verify_combine") for g in got), got
set_layer(0, sz.Q8_0)
stub.stub_fail_allocations_over(1 << 16)     # the EXL3 launches' buffers
fails("hipMalloc", lambda: set_layer(0, sz.EXL3(3)))
fails("hipMalloc", lambda: set_layer(1, sz.EXL3(3)))
launched(0, "q8_0")
fails("no experts set", lambda: layer(1))
stub.stub_fail_allocations_over(1 << 62)
for n in (0, 1):                             # the address table's copy, the table of EXL3 layers
    stub.stub_fail_copy_after(n)
    fails("hipMemcpyHtoD", lambda: set_layer(1, sz.EXL3(3)))
    stub.stub_fail_copy_after(-1)
    fails("no experts set", lambda: layer(1))
for l, ty in enumerate((sz.EXL3(4), sz.EXL3(3), sz.Q8_0, sz.EXL3(2))):
    set_layer(l, ty)
    launched(l, "q8_0" if ty == sz.Q8_0 else "exl3")
stub.stub_fail_copy_after(1)
fails("hipMemcpyHtoD", lambda: set_layer(1, sz.EXL3(2)))
stub.stub_fail_copy_after(-1)
fails("layer 1 has no experts set", lambda: s.verify_round(M, u, rl, sgl, y, hu, dr, out, 16))
launched(3, "exl3_2")
set_layer(1, sz.EXL3(2))
s.verify_round(M, u, rl, sgl, y, hu, dr, out, 16)
''')


@pytest.mark.parametrize("ty", ["sz.Q8_0", "sz.IQ3_S", "sz.F32", "sz.BF16"])
def test_a_product_over_no_columns_is_launched_as_one(stub, ty):
    """Rows of no columns are taken: every output is the empty sum, written by the kernel that takes a weight at a time."""
    stub(f"""
sz.matvec_cols({ty}, 256, 0, 100, 512, 0, 1024, 128, 3, 0, 0, 16)
got = taken()
assert [g[0] for g in got] == ["matvec_q8_0"] * 3 and [g[2][2:] for g in got] == [[1024 + 512 * j, 100, 0] for j in range(3)], got
""")


# bits (0.5 more: a half rate), inputs, columns, rows, the tiles a wave that are within 1.5 % of the fastest there
TILES = [(1, 5, 4096, 20480, 2), (1, 8, 2048, 40960, 2), (2, 5, 4096, 20480, 2), (2.5, 5, 2048, 40960, 2), (3, 5, 4096, 20480, 4), (4, 8, 2048, 40960, 4),
         (4, 5, 2048, 24576, 2), (1, 5, 4096, 14336, 4), (6, 8, 2048, 32768, 4), (4, 5, 4096, 18432, 2), (1, 5, 4096, 28672, 2), (2, 8, 4096, 28672, 8), (4, 5, 4096, 28672, 8),
         (2, 5, 2048, 65536, 4), (2, 8, 2048, 65536, 8), (4, 5, 8192, 16384, 8), (3, 8, 4096, 36864, 4), (1, 5, 8192, 22528, 8), (1, 5, 8192, 28672, 4), (4, 5, 8192, 28672, 4),
         (6, 5, 8192, 28672, 8), (4, 8, 4096, 67584, 8), (2, 5, 4096, 67584, 4), (4, 5, 8192, 32768, 8), (4, 8, 4096, 16512, 2), (4, 8, 2048, 65792, 4),
         (6, 8, 2048, 4096, 1), (6, 4, 2048, 4096, 1), (6, 8, 640, 4096, 2), (3.5, 8, 2048, 4096, 2), (4, 4, 4096, 20480, 2), (4, 1, 8192, 32768, 4)]


def test_the_tiles_of_a_projection(stub):
    """At the edges of the rule: what a call launches is what was fastest there."""
    stub(f"""
for bits, m, cols, rows, want in {TILES}:
    half, kb = bits % 1 > 0, int(bits)
    ty = sz.EXL3_HALF(kb) if half else sz.EXL3(kb)
    sz.matvec_cols(ty, 256, cols, rows, 512, cols, 1024, rows, m, 4096, sz.matvec_cols_scratch(ty, cols, rows, m), 16)
    (name, shape, _), finish = taken()
    kind = {{8: "", 4: "t4", 2: "t2", 1: "t1"}}[want] + ("w_" if m > 4 else "" if want == 8 else "_")
    assert name == "matvec_grouped_" + kind + ("exl3h_" if half else "exl3_") + str(kb), (bits, m, cols, rows, name)
    assert shape[:3] == (rows // (64 * want), -(-cols // 512), 1) and finish[0] == "exl3_finish_rows", (bits, m, cols, rows, shape)
""")
