"""The work a speculative-decoding engine hands this library, as cases with inputs, outputs, minimum work and tolerances.

An engine calls it in these ways, and each is a `kind` here:

  backend   one matrix-vector product on host buffers, the matrix resident under its key (GpuBackend.matvec)
  cols      dense projections on device buffers for the 1..8 rows of a decode or verify batch (matvec_cols), several in a row
  block     the router and the MoE block of several layers, a call a layer, as between attention layers (Session.moe_block_verify)
  round     the MoE layers, head, arg-max and acceptance of a whole verify round (Session.verify_round)
  prefill   a chunk of a prompt through one MoE layer (Session.moe_prefill_chunk)
  top       the head's 64 best logits of every row, handed to the sampler on the host (Session.head_top)
  hyper     the hyper-connection's read before and write after a sublayer (HyperConnection.read, hc_write)

Sizes are those of the repository's configurations (hidden 2048, 512 experts of 512, top-10, a vocabulary of 151936), tests
and checkpoints of the same kind with fewer, wider experts.  Weights are random in the formats' own value ranges.
"""
import math

import numpy as np
import torch

import shadow_engine_amd as sz
from shadow_engine_amd import synth, synth_device

DENSE = {"f32": sz.F32, "f16": sz.F16, "bf16": sz.BF16}
GGUF = {"q8_0": sz.Q8_0, "iq3_s": sz.IQ3_S}


def listed():
    return [
        # one expert's fused gate and up for one token through the host-side backend: the smallest call there is
        {"name": "backend-q8_0-1024x2048", "kind": "backend", "type": "q8_0", "cols": 2048, "rows": 1024},
        # a checkpoint's quantized projections for a batch of five, shapes that fill no tile evenly
        {"name": "cols-q8_0-5rows", "kind": "cols", "type": "q8_0", "cols": 3072, "rows": 8201, "m": 5, "count": 2},
        # the attention projections of an EXL3 checkpoint for a verify batch
        {"name": "cols-exl3_4-4rows", "kind": "cols", "type": "exl3_4", "cols": 2048, "rows": 4096, "m": 4, "count": 4},
        # plain decoding, no drafts: one token through eight layers
        {"name": "block-iq3_s-1row", "kind": "block", "type": "iq3_s", "hidden": 2048, "ff": 512, "experts": 512, "k": 10, "shared": True,
         "router": "bf16", "layers": 8, "m": 1},
        # the largest verify batch through layers with fewer, wider experts and no shared one
        {"name": "block-q8_0-8rows", "kind": "block", "type": "q8_0", "hidden": 2560, "ff": 768, "experts": 128, "k": 8, "shared": False,
         "router": "f32", "layers": 4, "m": 8},
        # an accepted token and three drafts through EXL3 layers, a call a layer
        {"name": "block-exl3_3-4rows", "kind": "block", "type": "exl3_3", "hidden": 2048, "ff": 512, "experts": 512, "k": 10, "shared": True,
         "router": "bf16", "layers": 6, "m": 4},
        # the full-depth verify round: mixed bit rates, about 30 GB of experts, a Q8_0 head
        {"name": "round-48layers-4rows", "kind": "round", "rates": "2,3,4", "hidden": 2048, "ff": 512, "experts": 512, "k": 10, "shared": True,
         "layers": 48, "m": 4, "head": "q8_0", "vocab": 151936},
        # a chunk of a prompt on int8 activations
        {"name": "prefill-iq3_s-512", "kind": "prefill", "type": "iq3_s", "hidden": 2048, "ff": 512, "experts": 512, "k": 10, "shared": False,
         "tokens": 512},
        # a short question
        {"name": "prefill-exl3_3-45", "kind": "prefill", "type": "exl3_3", "hidden": 2048, "ff": 512, "experts": 512, "k": 10, "shared": True,
         "tokens": 45},
        # a long document
        {"name": "prefill-exl3_4-4096", "kind": "prefill", "type": "exl3_4", "hidden": 2048, "ff": 512, "experts": 512, "k": 10, "shared": True,
         "tokens": 4096},
        # sampling from an EXL3 head
        {"name": "top-exl3_4-4rows", "kind": "top", "type": "exl3_4", "hidden": 2048, "vocab": 151936, "m": 4},
        # the residual streams around a block
        {"name": "hyper-bf16-4rows", "kind": "hyper", "type": "bf16", "hidden": 2048, "streams": 4, "rank": 320, "m": 4},
    ]


# ---- drawing cases ---------------------------------------------------------------------------------------------------------
def log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def log_step(rng, lo, hi, step):
    """A multiple of `step` in [lo, hi], spread over the logarithm."""
    return min(hi // step, max(-(-lo // step), round(log_int(rng, lo, hi) / step))) * step


def step_int(rng, lo, hi, step):
    return rng.randrange(lo // step, hi // step + 1) * step


def draw(rng):
    by_name = {c["name"]: c for c in listed()}
    deep, long = by_name["round-48layers-4rows"], by_name["prefill-exl3_4-4096"]
    while True:
        c = DRAW[rng.choice(sorted(DRAW))](rng)
        w = work(c)
        if (resident_bytes(c) <= 1.02 * resident_bytes(deep) and w["bytes"] <= work(deep)["bytes"] and
                w["flops"] <= work(long if c["kind"] == "prefill" else deep)["flops"]):
            return c


def draw_matrix(rng, types, rows_most):
    ty = rng.choice(types)
    rows, cols = log_int(rng, 128, rows_most), log_step(rng, 256, 8192, 256)
    if ty.startswith("exl3"):
        return {"type": ty, "cols": -(-cols // 128) * 128, "rows": -(-rows // 128) * 128}
    return {"type": ty, "cols": cols if ty == "iq3_s" else cols - 32 * rng.randrange(0, 4), "rows": rows}


def draw_moe(rng, types):
    ne = rng.choice([32, 60, 64, 128, 160, 256, 512])
    return {"type": rng.choice(types), "hidden": step_int(rng, 1024, 4096, 256), "ff": step_int(rng, 256, 1536, 256), "experts": ne,
            "k": rng.randrange(2, 13), "shared": rng.random() < 0.6}


def draw_backend(rng):
    return {"kind": "backend", **draw_matrix(rng, ["q8_0", "iq3_s", "exl3_3", "exl3_4"], 16384)}


def draw_cols(rng):
    return {"kind": "cols", **draw_matrix(rng, ["q8_0", "iq3_s", "bf16", "f16", "exl3_2", "exl3_3", "exl3_4", "exl3_5", "exl3_6"], 32768),
            "m": rng.randrange(1, 9), "count": rng.randrange(1, 5)}


def draw_block(rng):
    return {"kind": "block", **draw_moe(rng, ["q8_0", "iq3_s", "exl3_2", "exl3_3", "exl3_4", "exl3_2h"]), "router": rng.choice(["f32", "bf16"]),
            "layers": rng.randrange(2, 9), "m": rng.randrange(1, 9)}


def draw_round(rng):
    c = draw_moe(rng, ["exl3"])
    del c["type"]
    return {"kind": "round", **c, "rates": rng.choice(["2", "3", "4", "2,3,4", "3,4"]), "layers": log_int(rng, 4, 48), "m": rng.randrange(1, 9),
            "head": rng.choice(["q8_0", "exl3_4"]), "vocab": log_step(rng, 32000, 262144, 128)}


def draw_prefill(rng):
    c = draw_moe(rng, ["iq3_s", "exl3_2", "exl3_3", "exl3_4"])
    if c["type"] != "iq3_s":
        c["ff"] = rng.choice([256, 512])
    return {"kind": "prefill", **c, "tokens": log_int(rng, 16, 4096)}


def draw_top(rng):
    return {"kind": "top", "type": rng.choice(["q8_0", "exl3_3", "exl3_4", "exl3_5", "exl3_6"]), "hidden": step_int(rng, 1024, 4096, 256),
            "vocab": log_step(rng, 32000, 262144, 128), "m": rng.randrange(1, 9)}


def draw_hyper(rng):
    return {"kind": "hyper", "type": rng.choice(["bf16", "f16", "f32"]), "hidden": step_int(rng, 1024, 4096, 256), "streams": rng.choice([2, 3, 4]),
            "rank": step_int(rng, 64, 512, 4), "m": rng.randrange(1, 9)}


DRAW = {"backend": draw_backend, "cols": draw_cols, "block": draw_block, "round": draw_round, "prefill": draw_prefill, "top": draw_top, "hyper": draw_hyper}


# ---- sizes -----------------------------------------------------------------------------------------------------------------
def type_id(ty):
    if ty in DENSE or ty in GGUF:
        return DENSE.get(ty, GGUF.get(ty))
    return sz.EXL3_HALF(int(ty[5])) if ty.endswith("h") else sz.EXL3(int(ty[5:]))


def matrix_bytes(ty, cols, rows):
    if ty in DENSE:
        return cols * rows * (4 if ty == "f32" else 2)
    if ty in GGUF:
        return rows * (cols // 32 * 34 if ty == "q8_0" else cols // 256 * 110)
    return synth.exl3_blob_len(cols, rows, int(ty[5]), ty.endswith("h"))


def expert_bytes(c, ty):
    return 2 * matrix_bytes(ty, c["hidden"], c["ff"]) + matrix_bytes(ty, c["ff"], c["hidden"])


def layer_types(c):
    """The type of every layer of a round: as many of each rate as divide evenly, in a seeded order."""
    if c["kind"] != "round":
        return [c["type"]] * c.get("layers", 1)
    return ["exl3_%d" % r for r in synth_device.layer_rates(5, c["layers"], [int(r) for r in c["rates"].split(",")])]


def distinct(c, rows):
    """Distinct experts that `rows` tokens choose: expected for independent choices; with a prompt's skewed popularity, of a sample."""
    if c["kind"] == "prefill":
        logits = synth.zipf_router_logits(np.random.default_rng(1), rows, c["experts"])
        return int(np.unique(np.argpartition(-logits, c["k"] - 1, axis=1)[:, :c["k"]]).size)
    return c["experts"] * (1.0 - (1.0 - c["k"] / c["experts"]) ** rows)


def resident_bytes(c):
    if c["kind"] in ("block", "round", "prefill"):
        head = matrix_bytes(c["head"], c["hidden"], c["vocab"]) if c["kind"] == "round" else 0
        return head + sum((c["experts"] + 1) * expert_bytes(c, ty) for ty in layer_types(c))
    return 0


def work(c):
    kind = c["kind"]
    if kind in ("backend", "cols"):
        m, n = c.get("m", 1), c.get("count", 1)
        return {"bytes": n * (matrix_bytes(c["type"], c["cols"], c["rows"]) + 4 * m * (c["cols"] + c["rows"])), "flops": 2.0 * n * m * c["cols"] * c["rows"]}
    if kind in ("block", "round", "prefill"):
        m = c["tokens"] if kind == "prefill" else c["m"]
        d, pairs = distinct(c, m) + c["shared"], m * (c["k"] + c["shared"])
        types = layer_types(c)
        b = sum(d * expert_bytes(c, ty) for ty in types) + 4 * len(types) * m * 2 * c["hidden"]
        fl = len(types) * pairs * 6.0 * c["hidden"] * c["ff"]
        if kind == "block":
            b += len(types) * matrix_bytes(c["router"], c["hidden"], c["experts"] + c["shared"])
            fl += len(types) * m * 2.0 * c["hidden"] * (c["experts"] + c["shared"])
        else:
            b += 4 * len(types) * m * (c["experts"] + 1)
        if kind == "round":
            b += matrix_bytes(c["head"], c["hidden"], c["vocab"]) + 4 * m * c["hidden"]
            fl += 2.0 * m * c["hidden"] * c["vocab"]
        return {"bytes": b, "flops": fl}
    if kind == "top":
        return {"bytes": matrix_bytes(c["type"], c["hidden"], c["vocab"]) + 4 * c["m"] * (c["hidden"] + 128), "flops": 2.0 * c["m"] * c["hidden"] * c["vocab"]}
    ch = c["hidden"] * c["streams"]
    weights = ch * (2 * c["rank"] + c["streams"])
    return {"bytes": weights * (4 if c["type"] == "f32" else 2) + 4 * ch + 4 * c["m"] * (2 * ch + 2 * c["hidden"]), "flops": 2.0 * c["m"] * weights}


def tolerance(c):
    if c["kind"] == "prefill":
        return {"rel": 1e-3}                       # activations rounded to int8 codes or f16: the repository's own bound
    if c["kind"] == "top":
        return {"rel": 1e-5, "differ": 0.01}       # f32 sums; neighbours of the 64 whose logits agree to the last bits may change places
    return {"rel": 1e-5}                           # f32 sums over exactly decoded weights; token ids and counts do not differ


# ---- inputs ----------------------------------------------------------------------------------------------------------------
def generator(seed, salt=0):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed * 1000 + salt)
    return g


def normal(g, *shape):
    return torch.randn(shape, device="cuda", generator=g)


def matrix(seed, salt, ty, cols, rows):
    """A resident matrix as its stored bytes on the device."""
    key = seed * 1000 + salt
    if ty in DENSE:
        w = normal(generator(seed, salt), rows, cols) * 0.05
        return w if ty == "f32" else w.half() if ty == "f16" else w.bfloat16()
    if ty == "q8_0":
        return synth_device.q8_0_head(torch, key, rows, cols)
    if ty == "iq3_s":
        return iq3_s_rows(generator(seed, salt), rows * cols // 256)
    return synth_device.exl3_matrix(torch, key, cols, rows, int(ty[5]))


def iq3_s_rows(g, blocks):
    buf = torch.randint(0, 256, (blocks, 110), dtype=torch.uint8, device="cuda", generator=g)
    buf[:, :2] = (normal(g, blocks).abs() * 2e-4 + 1e-4).half().view(torch.uint8).reshape(blocks, 2)
    return buf.reshape(-1)


def experts(seed, salt, c, ty):
    """A layer's resident experts, the shared one last: (bytes, stride, gap)."""
    key, n = seed * 1000 + salt, c["experts"]
    if ty == "iq3_s":
        return (*synth_device.iq3_s_layer(torch, key, c["hidden"], c["ff"], n), 0)
    if ty == "q8_0":
        return synth_device.q8_0_head(torch, key, (n + 1) * 3 * c["ff"], c["hidden"]), expert_bytes(c, ty), 0
    if not ty.endswith("h"):
        return synth_device.exl3_layer(torch, key, c["hidden"], c["ff"], n, int(ty[5]), spaced=True)
    g = generator(seed, salt)
    parts = [(c["hidden"], c["ff"]), (c["hidden"], c["ff"]), (c["ff"], c["hidden"])]
    stride = -(-expert_bytes(c, ty) // 256) * 256
    buf = torch.randint(0, 256, (n + 1, stride), dtype=torch.uint8, device="cuda", generator=g)
    at = 0
    for cols, rows in parts:
        sign = torch.randint(0, 2, (n + 1, cols), device="cuda", generator=g)
        scale = 0.3 + torch.randint(0, 100, (n + 1, rows), device="cuda", generator=g) / 100.0
        for v in (1.0 - 2.0 * sign, scale):
            b = v.half().view(torch.uint8).reshape(n + 1, -1)
            buf[:, at:at + b.shape[1]] = b
            at += b.shape[1]
        buf[:, at:at + 4] = torch.tensor([1, 0, 0, 0], dtype=torch.uint8, device="cuda")
        at += matrix_bytes(ty, cols, rows) - 2 * (cols + rows)
    return buf.reshape(-1), stride, 0


def session(c, seed, types, vocab=0, head=None):
    s = sz.Session(c["hidden"], c.get("ff", 512), c.get("experts", 8), c.get("k", 2), len(types), vocab, 8)
    keep = []
    for l, ty in enumerate(types):
        buf, stride, gap = experts(seed, 10 + l, c, ty)
        shared = buf.data_ptr() + c["experts"] * stride if c["shared"] else 0
        s.set_layer(l, type_id(ty), buf.data_ptr(), stride, type_id(ty) if shared else 0, shared, gap=gap)
        keep.append(buf)
    if head:
        keep.append(matrix(seed, 1, head, c["hidden"], vocab))
        s.set_head(type_id(head), keep[-1].data_ptr())
    return s, keep


STREAM = []   # the engine's one stream: everything it asks for is queued there, in order


def prepare(c, seed):
    sz.init(0)
    if not STREAM:
        STREAM.append(sz.Stream())
    st = PREPARE[c["kind"]](c, seed)
    st["kind"], st["case"] = c["kind"], c
    torch.cuda.synchronize()
    return st


def prepare_backend(c, seed):
    w = matrix(seed, 1, c["type"], c["cols"], c["rows"]).cpu().numpy()
    rng = np.random.default_rng(seed)
    b = sz.GpuBackend()
    x = rng.standard_normal(c["cols"]).astype(np.float32)
    b.matvec(type_id(c["type"]), c["cols"], c["rows"], w, "w", x)      # the model's tensor is resident once the program is under way
    return {"backend": b, "type": type_id(c["type"]), "w": w, "x": x}


def prepare_cols(c, seed):
    g, ty, m = generator(seed), type_id(c["type"]), c["m"]
    n = sz.matvec_cols_scratch(ty, c["cols"], c["rows"], m)
    return {"type": ty, "w": [matrix(seed, 1 + i, c["type"], c["cols"], c["rows"]) for i in range(c["count"])],
            "x": normal(g, c["count"], m, c["cols"]), "y": torch.zeros(c["count"], m, c["rows"], device="cuda"),
            "scratch": torch.empty(max(n, 16), dtype=torch.uint8, device="cuda"), "scratch_bytes": n}


def prepare_block(c, seed):
    s, keep = session(c, seed, layer_types(c))
    for l in range(c["layers"]):
        w = matrix(seed, 100 + l, c["router"], c["hidden"], c["experts"])
        gate = matrix(seed, 200 + l, c["router"], c["hidden"], 1) if c["shared"] else None
        s.set_router(l, type_id(c["router"]), w.data_ptr(), type_id(c["router"]), gate.data_ptr() if c["shared"] else 0)
        keep += [w, gate]
    g = generator(seed)
    return {"session": s, "keep": keep, "u": normal(g, c["layers"], c["m"], c["hidden"]),
            "y": torch.zeros(c["layers"], c["m"], c["hidden"], device="cuda")}


def prepare_round(c, seed):
    s, keep = session(c, seed, layer_types(c), c["vocab"], c["head"])
    g, L, m = generator(seed), c["layers"], c["m"]
    st = {"session": s, "keep": keep, "u": normal(g, L, m, c["hidden"]), "rl": normal(g, L, m, c["experts"]),
          "sgl": normal(g, L, m), "head_u": normal(g, m, c["hidden"]), "y": torch.zeros(L, m, c["hidden"], device="cuda"),
          "drafts": torch.zeros(max(m - 1, 1), dtype=torch.int32, device="cuda"), "out": torch.zeros(2 + m, dtype=torch.int32, device="cuda")}
    # a drafter that is right twice: the head's own choices, the third draft another token
    ids = torch.zeros(8, dtype=torch.int32, device="cuda")
    torch.cuda.synchronize()
    s.head_argmax(m, st["head_u"].data_ptr(), ids.data_ptr(), STREAM[0].handle)
    STREAM[0].synchronize()
    st["drafts"][:m - 1] = ids[:m - 1]
    if m > 3:
        st["drafts"][2] = (ids[2] + 1) % c["vocab"]
    return st


def prepare_prefill(c, seed):
    s, keep = session(c, seed, [c["type"]])
    g, t = generator(seed), c["tokens"]
    rl = torch.from_numpy(synth.zipf_router_logits(np.random.default_rng(seed), t, c["experts"])).cuda()
    return {"session": s, "keep": keep, "x": normal(g, t, c["hidden"]), "rl": rl, "sgl": normal(g, t),
            "y": torch.zeros(t, c["hidden"], device="cuda")}


def prepare_top(c, seed):
    s, keep = session({**c, "shared": False}, seed, [], c["vocab"], c["type"])
    return {"session": s, "keep": keep, "u": normal(generator(seed), c["m"], c["hidden"])}


def prepare_hyper(c, seed):
    g, h, cs, ty = generator(seed), c["hidden"], c["streams"], type_id(c["type"])
    norm = 1.0 + 0.1 * normal(g, cs * h)
    down, up, inject = (matrix(seed, i, c["type"], cols, rows) for i, cols, rows in ((1, cs * h, c["rank"]), (2, c["rank"], cs * h), (3, cs * h, cs)))
    hc = sz.HyperConnection(h, cs, c["rank"], 1e-6, norm.data_ptr(), ty, down.data_ptr(), ty, up.data_ptr(), ty, inject.data_ptr())
    return {"hc": hc, "keep": [norm, down, up, inject], "r": normal(g, c["m"], cs * h), "u": torch.zeros(c["m"], h, device="cuda"),
            "y": 0.01 * normal(g, c["m"], h)}


PREPARE = {"backend": prepare_backend, "cols": prepare_cols, "block": prepare_block, "round": prepare_round, "prefill": prepare_prefill,
           "top": prepare_top, "hyper": prepare_hyper}


# ---- one pass --------------------------------------------------------------------------------------------------------------
def run(st):
    return RUN[st["kind"]](st, st["case"])


def run_backend(st, c):
    return st["backend"].matvec(st["type"], c["cols"], c["rows"], st["w"], "w", st["x"])


def run_cols(st, c):
    for w, x, y in zip(st["w"], st["x"], st["y"]):
        sz.matvec_cols(st["type"], w.data_ptr(), c["cols"], c["rows"], x.data_ptr(), c["cols"], y.data_ptr(), c["rows"], c["m"],
                       st["scratch"].data_ptr(), st["scratch_bytes"], STREAM[0].handle)
    return st["y"]


def run_block(st, c):
    for l in range(c["layers"]):
        st["session"].moe_block_verify(l, c["m"], st["u"][l].data_ptr(), st["y"][l].data_ptr(), STREAM[0].handle)
    return st["y"]


def run_round(st, c):
    st["session"].verify_round(c["m"], st["u"].data_ptr(), st["rl"].data_ptr(), st["sgl"].data_ptr(), st["y"].data_ptr(), st["head_u"].data_ptr(),
                               st["drafts"].data_ptr(), st["out"].data_ptr(), STREAM[0].handle)
    return st["y"], st["out"]


def run_prefill(st, c):
    st["session"].moe_prefill_chunk(0, c["tokens"], st["x"].data_ptr(), st["rl"].data_ptr(), st["sgl"].data_ptr(), st["y"].data_ptr(), STREAM[0].handle)
    return st["y"]


def run_top(st, c):
    return st["session"].head_top(c["m"], st["u"].data_ptr(), STREAM[0].handle)


def run_hyper(st, c):
    st["hc"].read(c["m"], st["r"].data_ptr(), st["u"].data_ptr(), STREAM[0].handle)
    sz.hc_write(st["r"].data_ptr(), st["hc"].gains, st["y"].data_ptr(), c["m"], c["hidden"], c["streams"], STREAM[0].handle)
    return st["u"], st["r"]


RUN = {"backend": run_backend, "cols": run_cols, "block": run_block, "round": run_round, "prefill": run_prefill, "top": run_top, "hyper": run_hyper}
