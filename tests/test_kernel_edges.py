"""The kernels' edges on the GPU: sizes at the ends of tiles, chunks and dispatch ranges, each against the CPU oracle."""
import numpy as np
import pytest

import oracle_lib as O
import shadow_engine_amd as sz
from shadow_engine_amd import synth, synth_device
from test_gpu_path import REL_L2, bits, build_layer, dense_matrix, dev, gguf_bound, gpu, oracle_layer, rel_l2  # noqa: F401 (gpu: the fixture)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ty,rows,cols", [(sz.Q8_0, 1, 32), (sz.Q8_0, 33, 288), (sz.Q8_0, 127, 736), (sz.Q8_0, 65, 1056), (sz.Q8_0, 8201, 256), (sz.Q8_0, 70, 4384),
                                          (sz.IQ3_S, 1, 256), (sz.IQ3_S, 129, 512), (sz.IQ3_S, 47, 1280), (sz.IQ3_S, 4200, 4352)])
@pytest.mark.parametrize("m", [1, 4, 5, 8])
def test_gguf_products_at_the_edges_of_tiles_and_chunks(gpu, ty, rows, cols, m):  # noqa: F811
    """Row counts around the 16-row tiles and past one tile a workgroup, rows shorter than a 256-column chunk, of one to more than
    sixteen chunks (two a wave), with a short last one, both widths of the input tile; inputs of very different sizes in one
    chunk; values past the last row stay untouched."""
    rng = np.random.default_rng(rows * 13 + cols + m)
    w = synth.q8_0_matrix(rng, rows, cols) if ty == sz.Q8_0 else synth.iq3_s_matrix(rng, rows, cols)
    x = rng.normal(size=(m, cols)).astype(np.float32) * np.exp2(rng.integers(-12, 12, size=(m, cols))).astype(np.float32)
    ys = rows + 5
    dw, dx = dev(gpu, w), dev(gpu, x)
    y = gpu.full((m, ys), 7.5, dtype=gpu.float32, device="cuda")
    sz.matvec_cols(ty, dw.data_ptr(), cols, rows, dx.data_ptr(), cols, y.data_ptr(), ys, m)
    gpu.cuda.synchronize()
    got = y.cpu().numpy()
    assert np.all(got[:, rows:] == 7.5)
    for j in range(m):
        want = O.matvec(ty, cols, rows, w, x[j])
        assert np.all(np.abs(got[j, :rows] - want) <= gguf_bound(ty, cols, rows, w, x[j]))
        assert np.linalg.norm(got[j, :rows] - want) <= REL_L2 * np.linalg.norm(want)
    # inputs that do not start on 16 bytes take the one-weight-at-a-time kernel
    d4 = gpu.empty(m * cols + 1, dtype=gpu.float32, device="cuda")
    d4[1:] = dx.flatten()
    sz.matvec_cols(ty, dw.data_ptr(), cols, rows, d4.data_ptr() + 4, cols, y.data_ptr(), ys, m)
    gpu.cuda.synchronize()
    for j in range(m):
        assert np.all(np.abs(y[j, :rows].cpu().numpy() - got[j, :rows]) <= 2 * gguf_bound(ty, cols, rows, w, x[j]))


@pytest.mark.parametrize("types,m", [((3, 0, 0), 4), ((0, 3, 0), 4), ((0, 0, 3), 1), ((0, 3, 0), 8), ((2, 0, 4, 0, 3), 4)])
def test_a_round_over_gguf_and_exl3_layers(gpu, types, m):  # noqa: F811
    """One or several EXL3 layers (the numbers: bits a weight) at any place among Q8_0 ones: a round gives the bits of the
    layer-by-layer calls, which the oracle checks, and the last layer's routing; so do its graph's replays."""
    rng = np.random.default_rng(sum(types) + m)
    hidden, ff, ne, k, vocab, L = 512, 256, 24, 3, 1024, len(types)
    s = sz.Session(hidden, ff, ne, k, L, vocab, 8)
    keep, want = [], []
    u, rl = rng.normal(size=(L, m, hidden)).astype(np.float32), rng.normal(size=(L, m, ne)).astype(np.float32)
    sgl, hu = rng.normal(size=(L, m)).astype(np.float32), rng.normal(size=(m, hidden)).astype(np.float32)
    for l, kb in enumerate(types):
        ty = sz.EXL3(kb) if kb else sz.Q8_0
        dbuf, stride, blobs, sh = build_layer(gpu, rng, ty, hidden, ff, ne, True)
        keep.append(dbuf)
        s.set_layer(l, ty, dbuf.data_ptr(), stride, ty, dbuf.data_ptr() + ne * stride)
        want.append(oracle_layer(ty, hidden, ff, k, blobs, sh, rl[l], sgl[l], u[l]))
    dhead = dev(gpu, synth.q8_0_matrix(rng, vocab, hidden))
    s.set_head(sz.Q8_0, dhead.data_ptr())
    du, drl, dsgl, dhu = dev(gpu, u), dev(gpu, rl), dev(gpu, sgl), dev(gpu, hu)
    drafts, out = gpu.zeros(8, dtype=gpu.int32, device="cuda"), gpu.zeros(10, dtype=gpu.int32, device="cuda")
    one = gpu.zeros((L, m, hidden), dtype=gpu.float32, device="cuda")
    for l in range(L):
        s.moe_layer_verify(l, m, du[l].data_ptr(), drl[l].data_ptr(), dsgl[l].data_ptr(), one[l].data_ptr())
    gpu.cuda.synchronize()
    one = one.cpu().numpy()
    for l in range(L):
        for j in range(m):
            assert rel_l2(one[l, j], want[l][0][j]) <= REL_L2
    stream, y = sz.Stream(), gpu.zeros((L, m, hidden), dtype=gpu.float32, device="cuda")
    for replay in range(3):
        y.zero_()
        gpu.cuda.synchronize()
        s.verify_round(m, du.data_ptr(), drl.data_ptr(), dsgl.data_ptr(), y.data_ptr(), dhu.data_ptr(), drafts.data_ptr(), out.data_ptr(), stream.handle)
        stream.synchronize()
        assert np.array_equal(bits(y.cpu().numpy()), bits(one)), f"replay {replay}"
        idx, _ = s.last_route(m, stream.handle)
        assert np.array_equal(idx, want[-1][1])


def products(gpu, ty, rows, cols, w, x):  # noqa: F811
    """W x_j for the rows of x, through matvec_cols."""
    m = x.shape[0]
    nsb = sz.matvec_cols_scratch(ty, cols, rows, m)
    dw, dx = dev(gpu, w), dev(gpu, x)
    scratch = gpu.empty(max(nsb, 16), dtype=gpu.uint8, device="cuda")
    y = gpu.zeros((m, rows), dtype=gpu.float32, device="cuda")
    sz.matvec_cols(ty, dw.data_ptr(), cols, rows, dx.data_ptr(), cols, y.data_ptr(), rows, m, scratch.data_ptr(), nsb)
    gpu.cuda.synchronize()
    return y.cpu().numpy()


def set_scales(ty, w, value):
    """The block scales (of an EXL3 blob of 512 inputs the output scales of 128) of w as one f16 value."""
    if ty >= 1000:
        w[1024:1024 + 256] = np.full(128, value, np.float16).view(np.uint8)
    else:
        w.reshape(-1, 34 if ty == sz.Q8_0 else 110)[:, :2] = np.array([value], np.float16).view(np.uint8)
    return w


@pytest.mark.parametrize("ty", [sz.Q8_0, sz.IQ3_S, sz.EXL3(3)])
@pytest.mark.parametrize("m", [1, 3, 8])
def test_products_of_subnormal_inputs(gpu, ty, m):  # noqa: F811
    """Inputs that are all subnormal, down to single units of 2^-149, are not lost.  Against f64 sums; the GGUF products of such
    inputs are exact up to f32 sums, an EXL3 one's transform rounds to multiples of 2^-149: nine additions and a scale for
    values of about 2^-130, under 2^-15 together, and as much again for its output side."""
    rng = np.random.default_rng(m)
    rows, cols = 128, 512
    w = synth.exl3_blob(rng, cols, rows, 3) if ty >= 1000 else synth.q8_0_matrix(rng, rows, cols) if ty == sz.Q8_0 else synth.iq3_s_matrix(rng, rows, cols)
    set_scales(ty, w, 16384.0)
    x = (rng.normal(size=(m, cols)) * 2.0 ** -130).astype(np.float32)
    if m > 2:
        x[2] = rng.integers(-3, 4, cols) * 2.0 ** -149 if ty < 1000 else 0.0
    assert np.abs(x).max() < 2.0 ** -126
    got = products(gpu, ty, rows, cols, w, x).astype(np.float64)
    for j in range(m):
        if ty >= 1000:
            want = O.exl3_matvec(cols, rows, 3, w, (x[j].astype(np.float64) * 2.0 ** 60).astype(np.float32)).astype(np.float64) * 2.0 ** -60
            assert np.linalg.norm(got[j] - want) <= 2.0 ** -14 * np.linalg.norm(want)
        else:
            want = O.dequantize(ty, w).reshape(rows, cols).astype(np.float64) @ x[j].astype(np.float64)
            assert np.linalg.norm(want) > 2.0 ** -126 and np.linalg.norm(got[j] - want) <= 1e-5 * np.linalg.norm(want)


@pytest.mark.parametrize("m", [1, 3, 8])
@pytest.mark.parametrize("cols", [256, 800, 4352])
def test_a_large_input_costs_the_others_no_bits(gpu, m, cols):  # noqa: F811
    """Inputs of four sizes from 2^-100 to 2^40 in every 32-block, and rows whose codes are zero but for the inputs of one size: every
    row's product is as good as f32 sums of its own terms, whatever lies beside them.  (512 terms and less a sum, in chunks:
    1e-5 of the sum of magnitudes is far above their rounding.)"""
    rng = np.random.default_rng(m + cols)
    rows = 96
    w = synth.q8_0_matrix(rng, rows, cols)
    size = rng.integers(0, 4, cols)
    size[:32:8] = [3, 0, 1, 2]
    codes = w.reshape(rows, cols // 32, 34)[:, :, 2:].reshape(rows, cols)
    codes[size[None, :] != (np.arange(rows) % 4)[:, None]] = 0
    w.reshape(rows, cols // 32, 34)[:, :, 2:] = codes.reshape(rows, cols // 32, 32)
    x = (rng.normal(size=(m, cols)) * np.array([1.0, 2.0 ** -50, 2.0 ** -100, 2.0 ** 40])[size]).astype(np.float32)
    if m > 2:
        x[2] = rng.normal(size=cols)             # an input without any such spread between others that have one
    got = products(gpu, sz.Q8_0, rows, cols, w, x).astype(np.float64)
    dense = O.dequantize(sz.Q8_0, w).reshape(rows, cols).astype(np.float64)
    for j in range(m):
        terms = dense * x[j].astype(np.float64)
        assert np.all(np.abs(got[j] - terms.sum(axis=1)) <= 1e-5 * np.abs(terms).sum(axis=1)), j


@pytest.mark.parametrize("ty", [sz.Q8_0, sz.IQ3_S])
@pytest.mark.parametrize("m", [1, 3, 8])
def test_an_infinite_input_gives_what_multiply_adds_give(gpu, ty, m):  # noqa: F811
    """One infinity: the sign of its weight's infinity, a NaN where that weight is zero; two that meet weights of opposite signs: a
    NaN; a NaN: a NaN; the inputs beside them in the batch, the largest floats among them, as without."""
    rng = np.random.default_rng(m)
    rows, cols = 48, 768
    w = synth.q8_0_matrix(rng, rows, cols) if ty == sz.Q8_0 else synth.iq3_s_matrix(rng, rows, cols)
    if ty == sz.Q8_0:
        w.reshape(rows, cols // 32, 34)[::3, 300 // 32, 2 + 300 % 32] = 0
    dense = O.dequantize(ty, w).reshape(rows, cols).astype(np.float64)
    assert ty == sz.Q8_0 or np.all(dense != 0.0)
    x = rng.normal(size=(m, cols)).astype(np.float32)
    x[0, 300] = np.inf
    if m > 2:
        x[1, [5, 300]] = -np.inf
        x[1, 6] = 3.0e38
    if m > 3:
        x[3, 700] = np.nan
        x[4, 300] = 1.0e38
        x[5] *= np.float32(1.0e-38)
    got = products(gpu, ty, rows, cols, w, x)
    with np.errstate(invalid="ignore", over="ignore"):
        for j in range(m):
            want = (dense * x[j].astype(np.float64)).sum(axis=1)
            assert np.array_equal(np.isnan(got[j]), np.isnan(want)), j
            ok = np.isfinite(want)
            assert np.array_equal(got[j][~ok & ~np.isnan(want)], want[~ok & ~np.isnan(want)]), j
            assert np.all(np.abs(got[j][ok] - want[ok]) <= 1e-5 * (np.abs(dense) * np.abs(x[j].astype(np.float64))).sum(axis=1)[ok]), j


@pytest.mark.parametrize("ty,h,cs,rank,m,size", [
    (sz.BF16, 2048, 4, 320, 4, 1.2e38), (sz.F32, 256, 2, 24, 8, 1.2e38), (sz.F16, 512, 4, 64, 1, 1e-30),   # streams near the largest f32, and tiny ones
    (sz.F16, 1024, 3, 64, 3, 1.0), (sz.BF16, 1280, 4, 64, 5, 1.0), (sz.F32, 1792, 4, 64, 8, 1.0),      # a row over 3, 5 and 7 waves
    (sz.BF16, 4096, 4, 128, 4, 1.0),                                                                   # rows that do not stay in registers
    (sz.F16, 100, 64, 24, 8, 1.0),                                                                     # a wave's span over several streams
    (sz.BF16, 9216, 64, 8, 8, 1.0)])                                                                   # rows in lots: seven, then one
def test_hyper_connection_at_its_edges(gpu, ty, h, cs, rank, m, size):  # noqa: F811
    """hc_read over sizes of streams, of the matrices' rows and of the values, against the oracle."""
    rng = np.random.default_rng(h + cs + m)
    ch, eps = h * cs, 1e-6 if size >= 1.0 else 0.0
    r = np.clip(rng.normal(size=(m, ch)) * size, -3.3e38, 3.3e38).astype(np.float32)
    nw = (1 + 0.1 * rng.normal(size=ch)).astype(np.float32)
    wd, wu, wi = dense_matrix(rng, ty, rank, ch), dense_matrix(rng, ty, ch, rank), dense_matrix(rng, ty, cs, ch)
    dr, dnw, dwd, dwu, dwi = dev(gpu, r), dev(gpu, nw), dev(gpu, wd), dev(gpu, wu), dev(gpu, wi)
    hc = sz.HyperConnection(h, cs, rank, eps, dnw.data_ptr(), ty, dwd.data_ptr(), ty, dwu.data_ptr(), ty, dwi.data_ptr())
    du = gpu.zeros((m, h), dtype=gpu.float32, device="cuda")
    hc.read(m, dr.data_ptr(), du.data_ptr())
    gpu.cuda.synchronize()
    u, g = du.cpu().numpy(), np.empty((m, cs), np.float32)
    sz.download(g, hc.gains)
    for j in range(m):
        wu_, wg_ = O.hc_read(r[j], h, cs, rank, eps, nw, (ty, wd), (ty, wu), (ty, wi))
        assert np.all(np.isfinite(wu_)) and rel_l2(u[j], wu_) <= 1e-5, rel_l2(u[j], wu_)
        assert np.allclose(g[j], wg_, rtol=1e-5, atol=1e-6)


@pytest.mark.parametrize("ty,h,cs,rank,m", [
    (sz.BF16, 2048, 4, 252, 4), (sz.BF16, 2048, 4, 256, 4),   # 256 workgroups of a row, and the first count with two
    (sz.F32, 1536, 4, 764, 8), (sz.F16, 1600, 3, 516, 1),     # three rows each, the last workgroups not full
    (sz.F16, 1152, 4, 2052, 3), (sz.BF16, 96, 4, 1028, 5),    # more than four each; four rows side by side, two of each after the other
    (sz.F32, 2052, 4, 516, 2), (sz.BF16, 4096, 4, 516, 1)])   # inputs that do not stay in registers: three each, two for one input
def test_hyper_connection_rows_of_a_workgroup(gpu, ty, h, cs, rank, m):  # noqa: F811
    """The rows a workgroup takes one after the other, at the counts where their number changes."""
    test_hyper_connection_at_its_edges(gpu, ty, h, cs, rank, m, 1.0)


@pytest.mark.parametrize("ty,h,cs,rank,m", [
    (sz.BF16, 4096, 4, 320, 5), (sz.F32, 2052, 4, 516, 8),    # more than 8192 columns: one row a workgroup for one input, several for more
    (sz.F16, 2304, 4, 1028, 3), (sz.BF16, 2048, 4, 320, 8),   # several for both; inputs that stay in registers
    (sz.F32, 4352, 64, 200, 8)])                              # inputs in lots: seven, then one
def test_hyper_connection_bits_do_not_depend_on_the_batch(gpu, ty, h, cs, rank, m):  # noqa: F811
    """hc_read of a row alone, in a batch of two and in one of m: the same bits."""
    rng = np.random.default_rng(h + cs + m)
    ch = h * cs
    r = rng.normal(size=(m, ch)).astype(np.float32)
    nw = (1 + 0.1 * rng.normal(size=ch)).astype(np.float32)
    wd, wu, wi = dense_matrix(rng, ty, rank, ch), dense_matrix(rng, ty, ch, rank), dense_matrix(rng, ty, cs, ch)
    dnw, dwd, dwu, dwi = dev(gpu, nw), dev(gpu, wd), dev(gpu, wu), dev(gpu, wi)
    hc = sz.HyperConnection(h, cs, rank, 1e-6, dnw.data_ptr(), ty, dwd.data_ptr(), ty, dwu.data_ptr(), ty, dwi.data_ptr())

    def read(rows):
        dr, du = dev(gpu, rows), gpu.zeros((len(rows), h), dtype=gpu.float32, device="cuda")
        hc.read(len(rows), dr.data_ptr(), du.data_ptr())
        gpu.cuda.synchronize()
        g = np.empty((len(rows), cs), np.float32)
        sz.download(g, hc.gains)
        return bits(du.cpu().numpy()), bits(g)

    u, g = read(r)
    for n in (1, 2):
        for j in range(0, m - n + 1, n):
            un, gn = read(r[j:j + n])
            assert np.array_equal(un, u[j:j + n]) and np.array_equal(gn, g[j:j + n]), (n, j)


@pytest.mark.parametrize("ty", [sz.F32, sz.F16, sz.BF16])
@pytest.mark.parametrize("rows,cols,m", [(9, 3072, 4), (5, 5000, 8), (6, 7168, 1), (17, 8192, 5), (3, 8196, 8), (1100, 9220, 3), (4, 20480, 4)])
def test_unquantized_rows_of_several_waves_and_longer(gpu, ty, rows, cols, m):  # noqa: F811
    """Rows over 3, 5, 7 and 8 waves of a workgroup, rows of more than 8192 columns, whose inputs do not stay in registers, and
    several passes of such rows a workgroup; every input has the bits of a launch of its own."""
    rng = np.random.default_rng(rows + cols + m)
    w, x = dense_matrix(rng, ty, rows, cols), rng.normal(size=(m, cols)).astype(np.float32)
    got = products(gpu, ty, rows, cols, w, x)
    for j in range(m):
        assert rel_l2(got[j], O.matvec(ty, cols, rows, w, x[j])) <= 1e-5
    assert np.array_equal(bits(products(gpu, ty, rows, cols, w, x[m - 1:])), bits(got[m - 1:]))


@pytest.mark.parametrize("m", [3, 8])
def test_a_round_of_more_layers_than_its_buffers_hold(gpu, m):  # noqa: F811
    """The EXL3 launches' sums are kept for as many layers as take 256 MiB (13 of this size): a round of 29 goes in three lots, whose
    bounds lie inside the runs of one bit rate, and gives the bits of the layer-by-layer calls, which use the buffers' start."""
    hidden, ff, ne, k, rates = 4096, 1536, 16, 16, [1, 2] * 14 + [2]
    per = 2 * 8 * (k + 1) * (hidden // 512) * ff * 4 + 8 * (k + 1) * (ff // 512) * hidden * 4
    assert (256 << 20) // per == 13
    L, g = len(rates), gpu.Generator(device="cuda")
    g.manual_seed(m)
    s = sz.Session(hidden, ff, ne, k, L, 1024, 8)
    bufs = {r: synth_device.exl3_layer(gpu, 7 + r, hidden, ff, ne, r, spaced=True) for r in (1, 2)}   # the layers differ by their inputs
    for l, r in enumerate(rates):
        buf, stride, gap = bufs[r]
        s.set_layer(l, sz.EXL3(r), buf.data_ptr(), stride, sz.EXL3(r), buf.data_ptr() + ne * stride, gap=gap)
    dhead = dev(gpu, synth.q8_0_matrix(np.random.default_rng(1), 1024, hidden))
    s.set_head(sz.Q8_0, dhead.data_ptr())
    u, rl, sgl, hu = (gpu.randn(sh, device="cuda", generator=g) for sh in ((L, m, hidden), (L, m, ne), (L, m), (m, hidden)))
    one, y = (gpu.zeros((L, m, hidden), dtype=gpu.float32, device="cuda") for _ in range(2))
    drafts, out = gpu.zeros(8, dtype=gpu.int32, device="cuda"), gpu.zeros(10, dtype=gpu.int32, device="cuda")
    gpu.cuda.synchronize()
    stream = sz.Stream()
    for l in range(L):
        s.moe_layer_verify(l, m, u[l].data_ptr(), rl[l].data_ptr(), sgl[l].data_ptr(), one[l].data_ptr(), stream.handle)
    for replay in range(3):
        s.verify_round(m, u.data_ptr(), rl.data_ptr(), sgl.data_ptr(), y.data_ptr(), hu.data_ptr(), drafts.data_ptr(), out.data_ptr(), stream.handle)
        stream.synchronize()
        assert gpu.all(gpu.isfinite(one)) and gpu.all(one.abs().amax(dim=2) > 0)
        assert gpu.equal(y.view(gpu.int32), one.view(gpu.int32)), f"replay {replay}"
        y.zero_()
        gpu.cuda.synchronize()


@pytest.mark.parametrize("ty", [sz.Q8_0, sz.BF16])
def test_products_over_no_columns_are_zero(gpu, ty):  # noqa: F811
    y = gpu.full((3, 128), 7.5, dtype=gpu.float32, device="cuda")
    sz.matvec_cols(ty, 0, 0, 100, 0, 0, y.data_ptr(), 128, 3)
    gpu.cuda.synchronize()
    assert gpu.all(y[:, :100] == 0.0) and gpu.all(y[:, 100:] == 7.5)


@pytest.mark.parametrize("kb,half", [(k, False) for k in range(1, 9)] + [(k, True) for k in range(1, 4)])
def test_every_tile_count_of_an_exl3_product_gives_the_same_bits(gpu, kb, half):  # noqa: F811
    """2, 4 and 8 column tiles a wave and both widths of the input tile, launched by name (which one a call takes follows from its
    size), on inputs that fill one block of 512 and a quarter of the next: the sums' order is the same, so are the bits; the
    oracle's values."""
    rng = np.random.default_rng(kb + 50 * half)
    cols, rows, m = 640, 1024, 8
    ty = sz.EXL3_HALF(kb) if half else sz.EXL3(kb)
    tag = ("exl3h_%d" if half else "exl3_%d") % kb
    w, x = synth.exl3_blob(rng, cols, rows, kb, half), rng.normal(size=(m, cols)).astype(np.float32)
    dw, dx = dev(gpu, w), dev(gpu, x)
    zs = (cols // 128 + 3) // 4
    P, U = sz.Arg.ptr, sz.Arg.u32

    def launched(form, ct, n):
        part = gpu.full((n, zs, rows), float("nan"), dtype=gpu.float32, device="cuda")
        y = gpu.zeros((n, rows), dtype=gpu.float32, device="cuda")
        sz.launch("matvec_grouped_" + form + tag, (rows // (64 * ct), zs, 1), (256, 1, 1), 0, 0,
                  [P(dw.data_ptr()), P(dx.data_ptr()), U(cols), P(part.data_ptr()), U(cols), U(rows), U(n)])
        sz.launch("exl3_finish_rows", (rows // 128, n, 1), (64, 1, 1), 0, 0, [P(part.data_ptr()), P(dw.data_ptr()), P(y.data_ptr()), U(rows), U(cols), U(rows)])
        gpu.cuda.synchronize()
        return y.cpu().numpy()

    first = launched("t2_", 2, 4)
    for j in range(4):
        assert rel_l2(first[j], O.exl3_matvec(cols, rows, kb, w, x[j], half=half)) <= 2e-6
    for form, ct in (("t4_", 4), ("", 8)):
        for n in (1, 3, 4):
            assert np.array_equal(bits(launched(form, ct, n)), bits(first[:n])), (form, n)
    for form, ct in (("t2w_", 2), ("t4w_", 4), ("w_", 8)):
        for n in (5, 8):
            got = launched(form, ct, n)
            assert np.array_equal(bits(got[:4]), bits(first)), (form, n)
            assert all(rel_l2(got[j], O.exl3_matvec(cols, rows, kb, w, x[j], half=half)) <= 2e-6 for j in range(4, n)), (form, n)


@pytest.mark.parametrize("m", [4, 8])
def test_a_deep_rounds_wide_tiles_give_the_bits_of_single_layers(gpu, m):  # noqa: F811
    """64 layers of one rate: enough waves for 8 column tiles each (at 4 rows 4 in the down launch), where a single layer takes 2.
    The bits agree in every layer, a sample of layers with the oracle."""
    rng = np.random.default_rng(m)
    hidden, ff, ne, k, L = 512, 512, 12, 4, 64
    s = sz.Session(hidden, ff, ne, k, L, 1024, 8)
    dbuf, stride, blobs, sh = build_layer(gpu, rng, sz.EXL3(3), hidden, ff, ne, True)      # the layers differ by their inputs
    for l in range(L):
        s.set_layer(l, sz.EXL3(3), dbuf.data_ptr(), stride, sz.EXL3(3), dbuf.data_ptr() + ne * stride)
    dhead = dev(gpu, synth.q8_0_matrix(rng, 1024, hidden))
    s.set_head(sz.Q8_0, dhead.data_ptr())
    u, rl = rng.normal(size=(L, m, hidden)).astype(np.float32), rng.normal(size=(L, m, ne)).astype(np.float32)
    sgl, hu = rng.normal(size=(L, m)).astype(np.float32), rng.normal(size=(m, hidden)).astype(np.float32)
    du, drl, dsgl, dhu = dev(gpu, u), dev(gpu, rl), dev(gpu, sgl), dev(gpu, hu)
    one, y = (gpu.zeros((L, m, hidden), dtype=gpu.float32, device="cuda") for _ in range(2))
    drafts, out = gpu.zeros(8, dtype=gpu.int32, device="cuda"), gpu.zeros(10, dtype=gpu.int32, device="cuda")
    gpu.cuda.synchronize()
    stream = sz.Stream()
    for l in range(L):
        s.moe_layer_verify(l, m, du[l].data_ptr(), drl[l].data_ptr(), dsgl[l].data_ptr(), one[l].data_ptr(), stream.handle)
    s.verify_round(m, du.data_ptr(), drl.data_ptr(), dsgl.data_ptr(), y.data_ptr(), dhu.data_ptr(), drafts.data_ptr(), out.data_ptr(), stream.handle)
    stream.synchronize()
    got = y.cpu().numpy()
    assert np.array_equal(bits(got), bits(one.cpu().numpy()))
    for l in (0, 31, 63):
        want, _, _ = oracle_layer(sz.EXL3(3), hidden, ff, k, blobs, sh, rl[l], sgl[l], u[l])
        assert all(rel_l2(got[l, j], want[j]) <= 2e-6 for j in range(m))


@pytest.mark.parametrize("ty", [sz.Q8_0, sz.IQ3_S])
@pytest.mark.parametrize("hidden,ff,ne,k,m,shared,finite", [
    (256, 256, 6, 2, 2, True, 6),       # one chunk a row: one wave a workgroup
    (2560, 768, 12, 4, 8, False, 12),   # experts of more than four tokens beside experts of one
    (4096, 512, 5, 3, 7, True, 5),      # 16 waves of 8 inputs: the most LDS a workgroup takes
    (4352, 1280, 4, 2, 3, True, 4),     # 17 chunks on 9 waves, tiles that do not divide among the workgroups
    (512, 4608, 4, 2, 5, True, 4),      # ff > 4096, and chunks on 9 waves in the down product
    (768, 256, 24, 16, 4, True, 11),    # the most experts a token, some of them masked: ranks without one
])
def test_gguf_layers_by_distinct_expert(gpu, monkeypatch, ty, hidden, ff, ne, k, m, shared, finite):  # noqa: F811
    """The layer on the matrix cores at the edges of its chunks, tiles and items, with a plan and pair by pair: the same bits, within
    2e-6 relative L2 of the oracle (f32 sums in another order: 2^-24 of a term for each of a few dozen partial sums)."""
    rng = np.random.default_rng(ty * 31 + hidden + m)
    dbuf, stride, blobs, sh = build_layer(gpu, rng, ty, hidden, ff, ne, shared)
    s = sz.Session(hidden, ff, ne, k, 1, 0, 8)
    s.set_layer(0, ty, dbuf.data_ptr(), stride, ty if shared else 0, dbuf.data_ptr() + ne * stride if shared else 0)
    u, logits, sgl = rng.normal(size=(m, hidden)).astype(np.float32), rng.normal(size=(m, ne)).astype(np.float32), rng.normal(size=m).astype(np.float32)
    logits[0, finite:] = -np.inf
    du, dl, dg = dev(gpu, u), dev(gpu, logits), dev(gpu, sgl)
    want, widx, ww = oracle_layer(ty, hidden, ff, k, blobs, sh, logits, sgl, u)
    outs = []
    for form in ("plan", "pairs"):
        monkeypatch.setenv("SHADOWZERO_GGUF_ITEMS", form)
        dy = gpu.zeros((m, hidden), dtype=gpu.float32, device="cuda")
        s.moe_layer_verify(0, m, du.data_ptr(), dl.data_ptr(), dg.data_ptr(), dy.data_ptr())
        gpu.cuda.synchronize()
        outs.append(dy.cpu().numpy())
        idx, w = s.last_route(m)
        assert np.array_equal(idx, widx) and np.allclose(w, ww, rtol=2e-6, atol=0)
        assert max(rel_l2(outs[-1][j], want[j]) for j in range(m)) <= 2e-6
    assert np.array_equal(bits(outs[0]), bits(outs[1]))


@pytest.mark.parametrize("ty,hidden,ff,ne,k,shared", [
    (sz.Q8_0, 1024, 256, 16, 4, False),         # the vector unit, a single token in two launches
    (sz.Q8_0, 3072, 256, 12, 2, True),          # rows of 96 units: three launches for a single token too
    (sz.Q8_0, 1280, 1024, 12, 2, True),         # just above the line: the matrix cores
    (sz.Q8_0, 2560, 768, 24, 8, False),
    (sz.IQ3_S, 2048, 512, 32, 10, True),        # below the line of the layers with two launches
    (sz.IQ3_S, 2048, 512, 32, 13, True),        # above it
    (sz.IQ3_S, 768, 1280, 8, 3, False),         # below the line of those without, rows of 24 and 40 units
    (sz.IQ3_S, 1792, 768, 16, 4, True),         # above it
    (sz.IQ3_S, 512, 4608, 6, 1, True),          # more than 4096 inputs of the down products
])
def test_a_gguf_layers_bits_do_not_depend_on_the_batch(gpu, ty, hidden, ff, ne, k, shared):  # noqa: F811
    """On both sides of every line of the choice between vector unit and matrix cores: a token's row has the same bits in batches of
    1 to 8 rows, within 2e-6 relative L2 of the oracle."""
    rng = np.random.default_rng(ty + hidden + ff + k)
    dbuf, stride, blobs, sh = build_layer(gpu, rng, ty, hidden, ff, ne, shared)
    s = sz.Session(hidden, ff, ne, k, 1, 0, 8)
    s.set_layer(0, ty, dbuf.data_ptr(), stride, ty if shared else 0, dbuf.data_ptr() + ne * stride if shared else 0)
    u, logits, sgl = rng.normal(size=(8, hidden)).astype(np.float32), rng.normal(size=(8, ne)).astype(np.float32), rng.normal(size=8).astype(np.float32)
    du, dl, dg = dev(gpu, u), dev(gpu, logits), dev(gpu, sgl)
    want, widx, _ = oracle_layer(ty, hidden, ff, k, blobs, sh, logits, sgl, u)
    first = None
    for m in range(8, 0, -1):
        y = gpu.zeros((m, hidden), dtype=gpu.float32, device="cuda")
        s.moe_layer_verify(0, m, du.data_ptr(), dl.data_ptr(), dg.data_ptr(), y.data_ptr())
        gpu.cuda.synchronize()
        got = y.cpu().numpy()
        assert np.array_equal(s.last_route(m)[0], widx[:m])
        if first is None:
            first = got
            assert max(rel_l2(got[j], want[j]) for j in range(8)) <= 2e-6
        assert np.array_equal(bits(got), bits(first[:m])), f"{m} rows"


@pytest.mark.parametrize("kb,tokens,hidden,ff", [(1, 129, 256, 256), (2, 40, 1024, 512), (4, 300, 256, 512), (5, 140, 512, 512), (6, 210, 256, 256), (7, 97, 256, 512),
                                                 (8, 260, 256, 512)] + [(kb, 8000, 256, 512) for kb in range(1, 9)])
def test_exl3_prefill_items_of_every_size(gpu, kb, tokens, hidden, ff):  # noqa: F811
    """Experts with few and many tokens (items of one tile to the most, the wide and the narrow form of the gate and up launch, the
    shortest streams) at every bit rate, a token of zeros, one of very large inputs, one whose products pass f32's range, and an
    expert whose gate is silent in one 128-block: that block's power of two is far from its neighbours'.  Every checked row within
    the chunk's 1e-3 of the oracle, or infinite and NaN where the oracle's is."""
    rng = np.random.default_rng(kb * 100 + tokens)
    ne, k, ty = 6, 2, sz.EXL3(kb)
    dbuf, stride, blobs, sh = build_layer(gpu, rng, ty, hidden, ff, ne, True)
    silent = 2 * hidden + 2 * (ff - 128)                     # the last 128 of gate's output scales
    for e in (0, 1):
        blobs[e][silent:silent + 256] = 0
        dbuf[e * stride + silent:e * stride + silent + 256] = 0
    s = sz.Session(hidden, ff, ne, k, 1, 0, 8)
    s.set_layer(0, ty, dbuf.data_ptr(), stride, ty, dbuf.data_ptr() + ne * stride)
    x = rng.normal(size=(tokens, hidden)).astype(np.float32)
    x[3], x[5], x[6] = 0.0, x[5] * np.float32(1e30), x[6] * np.float32(1e9)
    logits = rng.normal(size=(tokens, ne)).astype(np.float32) + np.log(np.array([40, 20, 8, 3, 1, 0.4], np.float32))
    sgl = rng.normal(size=tokens).astype(np.float32)
    dx, dl, dg = dev(gpu, x), dev(gpu, logits), dev(gpu, sgl)
    y = gpu.zeros((tokens, hidden), dtype=gpu.float32, device="cuda")
    s.moe_prefill_chunk(0, tokens, dx.data_ptr(), dl.data_ptr(), dg.data_ptr(), y.data_ptr())
    gpu.cuda.synchronize()
    got = y.cpu().numpy()
    rows = np.unique(np.r_[3, 4, 5, 6, rng.integers(0, tokens, 24), tokens - 1])
    want, _, _ = oracle_layer(ty, hidden, ff, k, blobs, sh, logits[rows], sgl[rows], x[rows])
    for i, j in enumerate(rows):
        if j == 3:
            assert not got[j].any()
        elif j == 5:
            assert np.array_equal(np.isfinite(got[j]), np.isfinite(want[i])) and not np.isfinite(want[i]).all()
        else:
            assert rel_l2(got[j], want[i]) <= 1e-3, (j, rel_l2(got[j], want[i]))


# What an expert's four 128-blocks of ff leave for the down product: the output scales of gate and up and the input scales of down
# whose product sets a block's size.  0, and 1e-22 as three of f16's subnormals, are silent beside any other.
BLOCK_SIZES = {"strong": (1, 45, 45), "huge": (3e4, 3e4, 3e4), "weak": (1, 1e-4, 1e-4), "weaker": (2e-7, 2e-7, 2e-7), "least": (6e-8, 6e-8, 6e-8), "ordinary": (1, 1, 1), "silent": (1, 0, 1)}


@pytest.mark.parametrize("kb", [2, 4, 7])
@pytest.mark.parametrize("tokens", [19, 700])
def test_exl3_prefill_blocks_of_any_size_beside_each_other(gpu, kb, tokens):  # noqa: F811
    """Every order of block sizes whose powers of two are far apart step by step, or only over several steps: the sums over ff stay
    in range, and every token's row is within the chunk's 1e-3 of the oracle (one expert a token, so that none hides another)."""
    rng = np.random.default_rng(kb * 1000 + tokens)
    orders = [("strong", "weak", "silent", "ordinary"), ("strong", "weaker", "silent", "ordinary"), ("huge", "weak", "least", "ordinary"), ("huge", "ordinary", "weaker", "silent"),
              ("least", "weak", "huge", "silent"), ("silent", "least", "ordinary", "strong"), ("strong", "silent", "weak", "silent"), ("weak", "silent", "silent", "weaker")]
    hidden, ff, ne, ty = 256, 512, len(orders), sz.EXL3(kb)
    dbuf, stride, blobs, _ = build_layer(gpu, rng, ty, hidden, ff, ne, False)
    gb, ub, _ = synth.expert_bytes(ty, hidden, ff)
    for e, order in enumerate(orders):
        for b, size in enumerate(order):
            for at, scale in zip((2 * hidden, gb + 2 * hidden, gb + ub), BLOCK_SIZES[size]):
                part = blobs[e][at + 256 * b:at + 256 * (b + 1)].view(np.float16)
                part[:] = (part.astype(np.float32) * scale).astype(np.float16)
        dbuf[e * stride:e * stride + blobs[e].size] = dev(gpu, blobs[e])
    s = sz.Session(hidden, ff, ne, 1, 1, 0, 8)
    s.set_layer(0, ty, dbuf.data_ptr(), stride, 0, 0)
    x, logits = rng.normal(size=(tokens, hidden)).astype(np.float32), np.full((tokens, ne), -9.0, np.float32)
    logits[np.arange(tokens), np.arange(tokens) % ne] = 9.0
    y = gpu.zeros((tokens, hidden), dtype=gpu.float32, device="cuda")
    dx, dl, dg = dev(gpu, x), dev(gpu, logits), dev(gpu, np.zeros(tokens, np.float32))
    s.moe_prefill_chunk(0, tokens, dx.data_ptr(), dl.data_ptr(), dg.data_ptr(), y.data_ptr())
    gpu.cuda.synchronize()
    got, rows = y.cpu().numpy(), np.r_[:16, tokens - 3:tokens]
    want, _, _ = oracle_layer(ty, hidden, ff, 1, blobs, None, logits[rows], np.zeros(rows.size, np.float32), x[rows])
    for i, j in enumerate(rows):
        assert rel_l2(got[j], want[i]) <= 1e-3, (orders[j % ne], rel_l2(got[j], want[i]))
    assert np.isfinite(got).all()


@pytest.mark.parametrize("kb", [3, 6])
@pytest.mark.parametrize("tokens", [19, 700])
def test_exl3_prefill_large_inputs_that_an_expert_scales_to_nothing(gpu, kb, tokens):  # noqa: F811
    """Inputs far above the others in channels whose scale is zero, f16's least, or a thousandth of the largest: what counts is the product, and the other channels keep
    their bits (within the chunk's 1e-3 of the oracle)."""
    rng = np.random.default_rng(kb * 1000 + tokens)
    hidden, ff, ne, k, ty = 512, 256, 4, 2, sz.EXL3(kb)
    dbuf, stride, blobs, _ = build_layer(gpu, rng, ty, hidden, ff, ne, False)
    gb, _, _ = synth.expert_bytes(ty, hidden, ff)
    for e in range(ne):
        for at in (0, gb):
            suh = blobs[e][at:at + 2 * hidden].view(np.float16)
            most = np.abs(suh.astype(np.float32)).max()
            suh[[3, 300, 7, 9]] = 0.0, 6e-8, most / 1024, most / 1200      # both sides of the line where launch 1 takes a pass for the products
        dbuf[e * stride:e * stride + blobs[e].size] = dev(gpu, blobs[e])
    s = sz.Session(hidden, ff, ne, k, 1, 0, 8)
    s.set_layer(0, ty, dbuf.data_ptr(), stride, 0, 0)
    x, logits = rng.normal(size=(tokens, hidden)).astype(np.float32), rng.normal(size=(tokens, ne)).astype(np.float32)
    x[0::4, 3] = 1e12
    x[1::4, 3] = -3.3e38
    x[2::4, 300] = 3e8
    x[3::8, 7], x[7::8, 9] = 2e5, 2e5
    y = gpu.zeros((tokens, hidden), dtype=gpu.float32, device="cuda")
    dx, dl, dg = dev(gpu, x), dev(gpu, logits), dev(gpu, np.zeros(tokens, np.float32))
    s.moe_prefill_chunk(0, tokens, dx.data_ptr(), dl.data_ptr(), dg.data_ptr(), y.data_ptr())
    gpu.cuda.synchronize()
    got, rows = y.cpu().numpy(), np.r_[:12, tokens - 4:tokens]
    want, _, _ = oracle_layer(ty, hidden, ff, k, blobs, None, logits[rows], np.zeros(rows.size, np.float32), x[rows])
    for i, j in enumerate(rows):
        assert rel_l2(got[j], want[i]) <= 1e-3, (j, rel_l2(got[j], want[i]))


@pytest.mark.parametrize("kb,hidden,ff,ne,k,shared,chunks", [
    (3, 1280, 512, 32, 2, False, (1400, 500, 60, 17)),        # items of up to 64 pairs, 32, 16; ten 128-blocks of hidden
    (2, 512, 256, 60, 8, False, (1300, 700, 100)),            # the same
    (4, 4096, 512, 16, 2, False, (260, 120, 20)),             # 32 blocks: shares of the rotation and of the down products
    (1, 256, 256, 40, 3, True, (1030, 200, 33, 1)),           # two blocks
    (2, 512, 512, 300, 8, False, (3000, 560, 130, 48)),       # both launches of eight waves, then of four
    (5, 512, 512, 140, 8, True, (2700, 500, 90)), (7, 512, 512, 140, 8, True, (2700, 500, 90)), (4, 256, 512, 16, 10, True, (2400, 250, 40)),
    (6, 768, 256, 32, 6, True, (400, 40)), (8, 768, 512, 32, 6, False, (400, 40))])
def test_exl3_prefill_bits_do_not_depend_on_the_chunk(gpu, kb, hidden, ff, ne, k, shared, chunks):  # noqa: F811
    """The first tokens of a chunk in chunks of their own, through the other forms and item lengths: the same bits, within the chunk's
    1e-3 of the oracle."""
    rng = np.random.default_rng(kb * 1000 + hidden)
    ty, most = sz.EXL3(kb), max(chunks)
    dbuf, stride, blobs, sh = build_layer(gpu, rng, ty, hidden, ff, ne, shared)
    s = sz.Session(hidden, ff, ne, k, 1, 0, 8)
    s.set_layer(0, ty, dbuf.data_ptr(), stride, ty if shared else 0, dbuf.data_ptr() + ne * stride if shared else 0)
    x, logits = rng.normal(size=(most, hidden)).astype(np.float32), synth.zipf_router_logits(rng, most, ne)
    sgl = rng.normal(size=most).astype(np.float32)
    dx, dl, dg = dev(gpu, x), dev(gpu, logits), dev(gpu, sgl)
    first = None
    for tokens in chunks:
        y = gpu.zeros((tokens, hidden), dtype=gpu.float32, device="cuda")
        s.moe_prefill_chunk(0, tokens, dx.data_ptr(), dl.data_ptr(), dg.data_ptr(), y.data_ptr())
        gpu.cuda.synchronize()
        got = y.cpu().numpy()
        if first is None:
            first = got
            rows = np.unique(np.r_[0, rng.integers(0, tokens, 10), tokens - 1])
            want, _, _ = oracle_layer(ty, hidden, ff, k, blobs, sh, logits[rows], sgl[rows], x[rows])
            for i, j in enumerate(rows):
                assert rel_l2(got[j], want[i]) <= 1e-3, (j, rel_l2(got[j], want[i]))
        assert np.array_equal(bits(got), bits(first[:tokens])), tokens


@pytest.mark.parametrize("hidden,ff", [(256, 256), (512, 768), (1024, 512)])
def test_iq3s_prefill_items_of_every_size(gpu, hidden, ff):  # noqa: F811
    """Experts with 1 to 130 tokens, at the edges of the tiles of 16 and the items of 64, over rows of one block (shorter than the
    stages in flight) and more; a token of zeros and one whose activations are close to f32's largest.  Every row within the chunk's
    1e-3 of the int8 oracle and, whatever the items' tiles, with the bits the token has in a chunk of its own; so has a chunk
    of the same tokens over and over, in which a workgroup takes several lots of rows."""
    rng = np.random.default_rng(hidden + ff)
    counts, ty = [1, 15, 16, 17, 31, 32, 33, 48, 49, 63, 64, 65, 80, 130], sz.IQ3_S
    ne = k = len(counts)
    tokens = max(counts)
    dbuf, stride, blobs, sh = build_layer(gpu, rng, ty, hidden, ff, ne, True)
    s = sz.Session(hidden, ff, ne, k, 1, 0, 8)
    s.set_layer(0, ty, dbuf.data_ptr(), stride, ty, dbuf.data_ptr() + ne * stride)
    x = rng.normal(size=(tokens, hidden)).astype(np.float32)
    x[2], x[4] = 0.0, x[4] / np.abs(x[4]).max() * np.float32(3e38)
    logits = rng.normal(size=(tokens, ne)).astype(np.float32)
    logits[np.arange(tokens)[:, None] >= np.array(counts)[None]] = -np.inf
    sgl = rng.normal(size=tokens).astype(np.float32)

    def chunk(x, logits, sgl):
        dx, dl, dg = dev(gpu, x), dev(gpu, logits), dev(gpu, sgl)
        y = gpu.zeros(x.shape, dtype=gpu.float32, device="cuda")
        s.moe_prefill_chunk(0, x.shape[0], dx.data_ptr(), dl.data_ptr(), dg.data_ptr(), y.data_ptr())
        gpu.cuda.synchronize()
        return y.cpu().numpy()

    got = chunk(x, logits, sgl)
    assert not got[2].any()
    for j in (0, 1, 3, 14, 15, 16, 40, 64, 100, tokens - 1):
        oi, ow = O.route(logits[j], k)
        wq, wd, _ = O.quantize_act(x[j], 32)
        want = np.zeros(hidden, np.float32)
        for e, w in zip(oi, ow):
            if e < ne:
                want = want + np.float32(w) * O.expert_int8(blobs[e], hidden, ff, wq, wd)[0]
        want = want + np.float32(O.lib().orc_sigmoid(float(sgl[j]))) * O.expert_int8(sh, hidden, ff, wq, wd)[0]
        assert rel_l2(got[j], want) <= REL_L2, (j, rel_l2(got[j], want))
    for j in (0, 2, 4, 15, 63, 64, 129):
        assert np.array_equal(bits(chunk(x[j:j + 1], logits[j:j + 1], sgl[j:j + 1])[0]), bits(got[j])), j
    reps = 1500                                              # long enough for several lots a workgroup
    big = chunk(np.resize(x, (reps, hidden)), np.resize(logits, (reps, ne)), np.resize(sgl, reps))
    assert np.array_equal(bits(big), bits(np.resize(got, (reps, hidden))))


@pytest.mark.parametrize("tokens,k", [(1024, 4), (1025, 4), (2049, 2), (1366, 3), (2731, 12), (16384, 2)])
def test_grouping_of_more_pairs_than_one_workgroup_lists(gpu, tokens, k):  # noqa: F811
    """4096 pairs, the first numbers beyond (a share of one run of 1024 pairs and a ragged one), some masked, and many: every token has
    the bits it has in chunks that one workgroup groups."""
    rng = np.random.default_rng(tokens + k)
    hidden, ff, ne, ty = 256, 256, 16, sz.IQ3_S
    dbuf, stride, _, _ = build_layer(gpu, rng, ty, hidden, ff, ne, True)
    s = sz.Session(hidden, ff, ne, k, 1, 0, 8)
    s.set_layer(0, ty, dbuf.data_ptr(), stride, ty, dbuf.data_ptr() + ne * stride)
    logits = synth.zipf_router_logits(rng, tokens, ne)
    logits[::7, :-k + 1] = -np.inf                           # fewer experts than k
    dx, dl, dg = dev(gpu, rng.normal(size=(tokens, hidden)).astype(np.float32)), dev(gpu, logits), dev(gpu, rng.normal(size=tokens).astype(np.float32))
    whole, cut = (gpu.zeros((tokens, hidden), dtype=gpu.float32, device="cuda") for _ in range(2))
    s.moe_prefill_chunk(0, tokens, dx.data_ptr(), dl.data_ptr(), dg.data_ptr(), whole.data_ptr())
    for t0 in range(0, tokens, 300):
        s.moe_prefill_chunk(0, min(300, tokens - t0), dx[t0:].data_ptr(), dl[t0:].data_ptr(), dg[t0:].data_ptr(), cut[t0:].data_ptr())
    gpu.cuda.synchronize()
    assert gpu.isfinite(whole).all() and np.array_equal(bits(whole.cpu().numpy()), bits(cut.cpu().numpy()))


@pytest.mark.parametrize("nob", [1, 2, 63, 64, 65, 130, 1187, 2048])
def test_the_64_best_from_the_blocks_largest(gpu, nob):  # noqa: F811
    """Fewer than 64 blocks of 128 logits to the most: random rows, rows whose best lie in few blocks (128 to 2048 as good as the 64th block's
    largest, and more), equal logits, zeros of both signs, infinities, NaN and nothing but -inf: values and ids as the
    oracle's sort gives them."""
    rng = np.random.default_rng(nob)
    n, rows = nob * 128, np.empty((8, nob * 128), np.float32)
    rows[0] = rng.normal(size=n)
    rows[1] = rng.normal(size=n) + 8 * (np.arange(n) // 128 % 97 == 5)
    rows[2] = rng.normal(size=n) * (1 + 30 * (np.arange(n) // 128 >= nob - 20))
    rows[3] = 1.25
    rows[4] = rng.integers(-3, 1, n) * 0.5
    rows[4, 3::11] = -0.0
    rows[5] = np.where(rng.random(n) < 0.01, np.nan, rng.normal(size=n))
    rows[5, rng.integers(0, n, 3)] = np.inf, -np.inf, np.inf
    rows[6] = -np.inf
    rows[6, rng.integers(0, n, 40)] = rng.normal(size=40)
    rows[7] = np.where(rng.random(n) < 0.5, np.nan, -np.inf)
    part = np.zeros((nob, 8, 2), np.uint32)
    clean = np.where(np.isnan(rows), -np.inf, rows).astype(np.float32).reshape(8, nob, 128)
    best = clean.argmax(axis=2)                              # the lowest id on ties
    part[:, :, 0] = bits(np.take_along_axis(clean, best[:, :, None], 2)[:, :, 0]).T
    part[:, :, 1] = (best + np.arange(nob) * 128).T
    dl, dp = dev(gpu, rows), dev(gpu, part.view(np.int32))
    out = gpu.zeros(8 * 128, dtype=gpu.int32, device="cuda")
    A = sz.Arg
    sz.launch("topk_blocks", (8, 1, 1), (1024, 1, 1), 0, 0, [A.ptr(dl.data_ptr()), A.u32(n), A.ptr(dp.data_ptr()), A.u32(nob), A.ptr(out.data_ptr())])
    gpu.cuda.synchronize()
    words = out.cpu().numpy().view(np.uint32).reshape(8, 128)
    for r in range(8):
        vals, ids = O.topk(rows[r], 64)
        assert np.array_equal(words[r, 64:], ids), f"row {r}"
        assert np.array_equal(words[r, :64], bits(vals)), f"row {r}"


@pytest.mark.parametrize("k,n,shared", [(1, 256, False), (3, 260, True), (10, 2048, True), (16, 1028, False)])
def test_chunk_combine_is_the_rows_combine(gpu, k, n, shared):  # noqa: F811
    """Four outputs a lane, the same bits: widths that leave the last workgroup part empty, tokens with fewer experts than k
    (whose other rows hold NaN), with and without the shared expert's row."""
    rng = np.random.default_rng(n + k)
    tokens = 7
    cnt = rng.integers(0, k + 1, tokens).astype(np.int32)
    cnt[0] = k
    eo = rng.normal(size=(tokens, k, n)).astype(np.float32)
    eo[np.arange(k)[None] >= cnt[:, None]] = np.nan
    bufs = [dev(gpu, a) for a in (eo, rng.random((tokens, k)).astype(np.float32), rng.normal(size=(tokens, n)).astype(np.float32), rng.normal(size=tokens).astype(np.float32), cnt)]
    A = sz.Arg
    ys = []
    for name, width, grid, block in (("moe_combine_qwen_rows", n, -(-n // 256), 256), ("prefill_combine", n // 4, -(-n // 256), 64)):
        y = gpu.full((tokens + 1, n), 7.0, dtype=gpu.float32, device="cuda")
        e, w, s, g, c = (b.data_ptr() for b in bufs)
        sz.launch(name, (grid, tokens, 1), (block, 1, 1), 0, 0, [A.ptr(y.data_ptr()), A.ptr(e), A.ptr(w), A.ptr(s if shared else 0), A.ptr(g), A.ptr(c), A.u32(width), A.u32(k)])
        gpu.cuda.synchronize()
        ys.append(y.cpu().numpy())
    assert np.isfinite(ys[0]).all() and (ys[0][tokens] == 7.0).all()
    assert np.array_equal(bits(ys[0]), bits(ys[1]))


@pytest.mark.parametrize("zs", [1, 4, 5, 8, 9, 16, 17, 21, 33])
def test_finish_adds_any_number_of_partials(gpu, zs):  # noqa: F811
    """exl3_finish_rows: sums of 1 to 33 partials (an input's 512 and a rest of 128), three rows of two output blocks, against
    64 bits.  zs - 1 additions, seven levels of the transform and its factor, a product: no more than zs + 9 roundings of 2^-24 of the
    magnitudes that go in."""
    rng = np.random.default_rng(zs)
    in_f, out_f, m = 512 * (zs - 1) + 128, 256, 3
    part = rng.normal(size=(m, zs, out_f)).astype(np.float32)
    svh = rng.normal(size=out_f).astype(np.float16)
    w = np.concatenate([rng.integers(0, 256, 2 * in_f).astype(np.uint8), svh.view(np.uint8)])
    dp, dw = dev(gpu, part), dev(gpu, w)
    y = gpu.zeros((m, out_f + 4), dtype=gpu.float32, device="cuda")
    A = sz.Arg
    sz.launch("exl3_finish_rows", (out_f // 128, m, 1), (64, 1, 1), 0, 0, [A.ptr(dp.data_ptr()), A.ptr(dw.data_ptr()), A.ptr(y.data_ptr()), A.u32(out_f + 4), A.u32(in_f), A.u32(out_f)])
    gpu.cuda.synchronize()
    h = np.ones((1, 1))
    while len(h) < 128:
        h = np.block([[h, h], [h, -h]])
    sums, mags = part.astype(np.float64).sum(1).reshape(m, 2, 128), np.abs(part.astype(np.float64)).sum((1,)).reshape(m, 2, 128).sum(2, keepdims=True)
    want = (sums @ h / np.sqrt(128)).reshape(m, out_f) * svh
    bound = np.broadcast_to((zs + 9) * 2.0**-24 * mags / np.sqrt(128), (m, 2, 128)).reshape(m, out_f) * np.abs(svh.astype(np.float64))
    assert (np.abs(y.cpu().numpy()[:, :out_f] - want) <= bound).all()


@pytest.mark.parametrize("kb,half", [(6, False), (7, False), (8, False), (3, True)])
@pytest.mark.parametrize("cols", [256, 640, 768, 2048])
def test_small_projections_above_five_bits(gpu, kb, half, cols):  # noqa: F811
    """One column tile a wave where the inputs come in 256s, two elsewhere (and at half rates): blocks of 512 inputs that are whole, a half and a quarter.  The oracle's
    values, and a row's bits whatever the rows beside it."""
    rng = np.random.default_rng(cols + kb)
    rows = 384
    ty = sz.EXL3_HALF(kb) if half else sz.EXL3(kb)
    w, x = synth.exl3_blob(rng, cols, rows, kb, half), rng.normal(size=(8, cols)).astype(np.float32)
    first = None
    for m in (1, 4, 5, 8):
        got = cols_call(gpu, ty, dev(gpu, w), cols, rows, x[:m])
        first = got if first is None else first
        assert np.array_equal(bits(got[:1]), bits(first[:1])), m
    for j in range(8):
        assert rel_l2(got[j], O.exl3_matvec(cols, rows, kb, w, x[j], half=half)) <= 2e-6, j


def cols_call(gpu, ty, dw, cols, rows, x):  # noqa: F811
    m, dx = len(x), dev(gpu, x)
    y = gpu.full((m, rows), float("nan"), dtype=gpu.float32, device="cuda")
    n = sz.matvec_cols_scratch(ty, cols, rows, m)
    scratch = gpu.empty(n, dtype=gpu.uint8, device="cuda")
    sz.matvec_cols(ty, dw.data_ptr(), cols, rows, dx.data_ptr(), cols, y.data_ptr(), rows, m, scratch.data_ptr(), n)
    gpu.cuda.synchronize()
    return y.cpu().numpy()


def exl3_columns(w, cols, rows, kb, at):
    """The blob of the 128 outputs from `at` on of an EXL3 matrix (host bytes): their scales and, of every 16 inputs, their eight tiles."""
    tiles = w[2 * (cols + rows) + 4:].reshape(cols // 16, rows // 16, 32 * kb)[:, at // 16:at // 16 + 8]
    return np.concatenate([w[:2 * cols], w[2 * (cols + at):2 * (cols + at + 128)], w[2 * (cols + rows):2 * (cols + rows) + 4], tiles.ravel()])


@pytest.mark.parametrize("kb", [2, 6])
@pytest.mark.parametrize("cols,rows", [(2048, 24576), (2048, 24704), (2048, 25088), (4096, 16384), (4096, 16512), (4096, 20480), (4096, 28672), (4096, 32768), (4096, 33280), (8192, 22528)])
def test_large_projections_for_more_than_four_inputs(gpu, cols, rows, kb):  # noqa: F811
    """The sizes at which a projection's tile count changes for more than four inputs, and rows that fill no wider workgroup: a row's bits are those of the calls
    of up to four, which choose by another rule; the first, a middle and the last block of 128 outputs are the oracle's, at a rate whose weights take one window and at
    one of two."""
    g = gpu.Generator(device="cuda")
    g.manual_seed(cols + rows)
    ty, dw = sz.EXL3(kb), synth_device.exl3_matrix(gpu, cols + rows, cols, rows, kb)
    x = gpu.randn((8, cols), device="cuda", generator=g).cpu().numpy()
    few = np.concatenate([cols_call(gpu, ty, dw, cols, rows, x[j:j + 4]) for j in (0, 4)])
    assert np.isfinite(few).all() and (np.abs(few).max(axis=1) > 0).all()
    for m in (5, 8):
        assert np.array_equal(bits(cols_call(gpu, ty, dw, cols, rows, x[:m])), bits(few[:m])), m
    w = dw.cpu().numpy()
    for at in (0, rows // 256 * 128, rows - 128):
        block = exl3_columns(w, cols, rows, kb, at)
        for j in (0, 7):
            assert rel_l2(few[j, at:at + 128], O.exl3_matvec(cols, 128, kb, block, x[j])) <= 2e-6, (at, j)


DOWN_FORMS = {4: (("t2_", 2), ("t4_", 4), ("", 8)), 8: (("t2w_", 2), ("t4w_", 4), ("w_", 8))}


@pytest.mark.parametrize("kb,half", [(k, False) for k in range(1, 9)] + [(k, True) for k in range(1, 4)])
@pytest.mark.parametrize("hidden,m", [(2560, 4), (4608, 8), (4608, 3), (2560, 6)])
def test_every_form_of_the_down_launch_of_more_than_four_partials(gpu, kb, half, hidden, m):  # noqa: F811
    """Gate and up sums of 5 and 9 partials through the kernels that ask for eight at once and those that ask for four, every tile count, launched by name on what
    a layer's call left behind (its plan and its sums): the same additions in the same order, so the same bits, in every pair's row.  The
    layer's own output is the oracle's."""
    rng = np.random.default_rng(100 * kb + hidden + m + half)
    ff, ne, k = 768, 6, 3
    ty = sz.EXL3_HALF(kb) if half else sz.EXL3(kb)
    tag = ("exl3h_%d" if half else "exl3_%d") % kb
    dbuf, stride, blobs, sh = build_layer(gpu, rng, ty, hidden, ff, ne, True)
    s = sz.Session(hidden, ff, ne, k, 1, 0, 8)
    shared = dbuf.data_ptr() + ne * stride
    s.set_layer(0, ty, dbuf.data_ptr(), stride, ty, shared)
    u, rl, sgl = rng.normal(size=(m, hidden)).astype(np.float32), rng.normal(size=(m, ne)).astype(np.float32), rng.normal(size=m).astype(np.float32)
    du, drl, dsgl, y = dev(gpu, u), dev(gpu, rl), dev(gpu, sgl), gpu.zeros((m, hidden), dtype=gpu.float32, device="cuda")
    sz.ktime_begin("verify_")
    s.moe_layer_verify(0, m, du.data_ptr(), drl.data_ptr(), dsgl.data_ptr(), y.data_ptr())
    gpu.cuda.synchronize()
    names = sz.ktime_end()
    assert "verify_plan_exl3" in names and "verify_down_x_" + ("t2w_" if m > 4 else "t2_") + tag in names, names
    want, _, _ = oracle_layer(ty, hidden, ff, k, blobs, sh, rl, sgl, u)
    assert all(rel_l2(y[j].cpu().numpy(), want[j]) <= 2e-6 for j in range(m))

    plan, sums = sz.lib().sz_session_buffer(s._h, 0), sz.lib().sz_session_buffer(s._h, 1)
    zd, part = -(-ff // 512), synth.expert_bytes(ty, hidden, ff)[0]
    ioff = -(-(2 * m * k * 4 + m * 4) // 16) * 16              # the items behind [ids | weights | counts]
    P, U, U64 = sz.Arg.ptr, sz.Arg.u32, sz.Arg.u64
    first = None
    for kind in ("verify_down_", "verify_down_x_"):
        for form, ct in DOWN_FORMS[8 if m > 4 else 4]:
            dn = gpu.full((m * (k + 1), zd, hidden), float("nan"), dtype=gpu.float32, device="cuda")
            sz.launch(kind + form + tag, (hidden // (64 * ct), m * k + 2, zd), (256, 1, 1), 0, 0,
                      [P(drl.data_ptr()), P(0), U64(dbuf.data_ptr()), U64(stride), U64(shared), U(part), U(0), P(plan), P(plan), U(0), U(ioff), P(sums), P(dn.data_ptr()),
                       U(ne), U(k), U(m), U(hidden), U(ff)])
            gpu.cuda.synchronize()
            got = bits(dn.cpu().numpy())
            first = got if first is None else first
            assert np.isfinite(dn.cpu().numpy()).all() and np.array_equal(got, first), (kind, form)


@pytest.mark.parametrize("ty", [sz.EXL3(3), sz.EXL3_HALF(2)])
@pytest.mark.parametrize("m,L,form", [(4, 8, "t4_"), (4, 32, ""), (8, 4, "t4w_"), (8, 16, "w_")])
def test_rounds_of_more_than_four_partials_take_wider_tiles(gpu, ty, m, L, form):  # noqa: F811
    """Layers of 2560 inputs, one run as a round's launch takes them: enough workgroups for 4 and 8 column tiles a wave of the down products.  A sample
    of the layers with the oracle."""
    rng = np.random.default_rng(m + L)
    hidden, ff, ne, k = 2560, 256, 6, 3
    s = sz.Session(hidden, ff, ne, k, L, 1024, 8)
    s.set_graph(False)
    dbuf, stride, blobs, sh = build_layer(gpu, rng, ty, hidden, ff, ne, True)      # the layers differ by their inputs
    for l in range(L):
        s.set_layer(l, ty, dbuf.data_ptr(), stride, ty, dbuf.data_ptr() + ne * stride)
    dhead = dev(gpu, synth.q8_0_matrix(rng, 1024, hidden))
    s.set_head(sz.Q8_0, dhead.data_ptr())
    u, rl = rng.normal(size=(L, m, hidden)).astype(np.float32), rng.normal(size=(L, m, ne)).astype(np.float32)
    sgl, hu = rng.normal(size=(L, m)).astype(np.float32), rng.normal(size=(m, hidden)).astype(np.float32)
    du, drl, dsgl, dhu = dev(gpu, u), dev(gpu, rl), dev(gpu, sgl), dev(gpu, hu)
    y = gpu.zeros((L, m, hidden), dtype=gpu.float32, device="cuda")
    drafts, out = gpu.zeros(8, dtype=gpu.int32, device="cuda"), gpu.zeros(10, dtype=gpu.int32, device="cuda")
    sz.ktime_begin("verify_down_")
    s.verify_round(m, du.data_ptr(), drl.data_ptr(), dsgl.data_ptr(), y.data_ptr(), dhu.data_ptr(), drafts.data_ptr(), out.data_ptr())
    gpu.cuda.synchronize()
    names = sz.ktime_end()
    assert list(names) == ["verify_down_x_" + form + ("exl3h_2" if ty == sz.EXL3_HALF(2) else "exl3_3")], names
    got = y.cpu().numpy()
    for l in (0, L // 2, L - 1):
        want, _, _ = oracle_layer(ty, hidden, ff, k, blobs, sh, rl[l], sgl[l], u[l])
        assert all(rel_l2(got[l, j], want[j]) <= 2e-6 for j in range(m)), l


@pytest.mark.parametrize("hidden,over", [(1024, 246724), (2048, 123362), (4096, 61681)])
@pytest.mark.parametrize("m", [1, 8])
def test_a_q8_0_head_about_as_large_as_the_last_level(gpu, hidden, over, m):  # noqa: F811
    """256 MiB, from where on a head is read past the caches, and a row less, which is not: the logits' bits are those of the head's two parts, and the ids
    their arg-max."""
    x = gpu.randn((m, hidden), device="cuda", generator=gpu.Generator(device="cuda").manual_seed(hidden))
    w = synth_device.q8_0_head(gpu, hidden, over, hidden)
    rb = hidden // 32 * 34
    assert over * rb >= 256 << 20 > (over - 1) * rb

    def logits(first, rows):
        s = sz.Session(hidden, 256, 8, 2, 0, rows, 8)
        s.set_head(sz.Q8_0, w.data_ptr() + first * rb)
        out, ids = gpu.full((m, rows), float("nan"), device="cuda"), gpu.zeros(m, dtype=gpu.int32, device="cuda")
        s.head_logits(m, x.data_ptr(), out.data_ptr())
        s.head_argmax(m, x.data_ptr(), ids.data_ptr())
        gpu.cuda.synchronize()
        assert gpu.equal(out.argmax(dim=1).int(), ids)
        return out

    cut = over // 2 // 16 * 16                               # 16-byte aligned, as a head has to be
    parts = gpu.cat([logits(0, cut), logits(cut, over - cut)], dim=1)
    assert gpu.isfinite(parts).all()
    for rows in (over, over - 1):
        assert gpu.equal(logits(0, rows), parts[:, :rows]), rows


@pytest.mark.parametrize("kb,hidden,blocks", [(3, 2048, 2731), (4, 2048, 2049), (8, 4096, 513)])
def test_an_exl3_head_about_as_large_as_the_last_level(gpu, kb, hidden, blocks):  # noqa: F811
    """A head just above 256 MiB, which is read past the caches, and one of the same blocks but the last, which is not: the same bits and ids; the last
    block is the oracle's."""
    m, rows = 5, 128 * blocks
    assert hidden * rows * kb // 8 > 256 << 20 >= hidden * (rows - 128) * kb // 8
    blob = synth_device.exl3_matrix(gpu, kb, hidden, rows, kb)
    x = gpu.randn((m, hidden), device="cuda", generator=gpu.Generator(device="cuda").manual_seed(kb))
    at, tiles = 2 * (hidden + rows), blob[2 * (hidden + rows) + 4:].view(hidden // 16, rows // 16, 32 * kb)
    smaller = gpu.cat([blob[:at - 256], blob[at:at + 4], tiles[:, :rows // 16 - 8].reshape(-1)])

    def run(w, n):
        s = sz.Session(hidden, 256, 8, 2, 0, n, 8)
        s.set_head(sz.EXL3(kb), w.data_ptr())
        out, ids = gpu.full((m, n), float("nan"), device="cuda"), gpu.zeros(m, dtype=gpu.int32, device="cuda")
        sz.ktime_begin("head_exl3_")
        s.head_logits(m, x.data_ptr(), out.data_ptr())
        s.head_argmax(m, x.data_ptr(), ids.data_ptr())
        gpu.cuda.synchronize()
        names = sz.ktime_end()
        assert list(names) == ["head_exl3_" + ("past_" if n == rows else "") + str(kb)], names
        assert gpu.isfinite(out).all() and gpu.equal(out.argmax(dim=1).int(), ids)
        return out

    whole = run(blob, rows)
    assert gpu.equal(run(smaller, rows - 128), whole[:, :rows - 128])
    w = blob.cpu().numpy()
    last = exl3_columns(w, hidden, rows, kb, rows - 128)
    for j in (0, m - 1):
        assert rel_l2(whole[j, rows - 128:].cpu().numpy(), O.exl3_matvec(hidden, 128, kb, last, x[j].cpu().numpy())) <= REL_L2
