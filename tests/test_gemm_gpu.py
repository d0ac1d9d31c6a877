"""Parity of quant_rows_i8 (bit-exact) and the W8A16 fc1 GEMM + SwiGLU epilogue (bf16 at 1e-2) with the oracle."""
import re
from pathlib import Path

import numpy as np
import pytest
import torch

import mako_h3 as mh
import oracle as orc
from helpers import (assert_close, bits_to_f64, check_gemm_full, diff, from_bits, nan_filled, randn_bf16_bits,
                     to_bits)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", ["bf16", "f32"])
@pytest.mark.parametrize("rows,cols", [(1, 16), (7, 5120), (300, 208), (5, 2048), (6, 4096), (3, 8192), (3, 8208),
                                       (4, 13824), (2, 14336), (3, 14352), (2, 27648)])
def test_quant_rows_i8_bit_exact(dev, dtype, rows, cols):
    """Widths up to 14,336 keep the row in registers (2, 4, 8 or 14 chunks of 16 a lane); wider rows take the two-read
    path. The row's last element carries its maximum in one row, so a dropped tail chunk changes the scale."""
    rng = np.random.default_rng(rows + cols)
    if dtype == "bf16":
        w = randn_bf16_bits(rng, (rows, cols), 0.02)
        w[0, :] = 0                                        # an all-zero row: scale 0, q 0
        if rows > 1:
            w[1, -1] = 0x3F80                              # 1.0 at the row's last element: its maximum
        tw = from_bits(w, dev)
    else:
        w = (rng.standard_normal((rows, cols)) * 0.02).astype(np.float32)
        w[0, :] = 0
        if rows > 1:
            w[1, 3] = -1.0                                 # the row maximum on the negative side
        tw = torch.from_numpy(w).to(dev)
    q, s = mh.quant_rows_i8(tw)
    wq, ws = orc.quant_rows_i8(w)
    assert (s.cpu().numpy() == ws).all()
    assert (q.cpu().numpy() == wq).all()


@pytest.mark.parametrize("cols", [208, 5120, 13824, 27648])
def test_quant_rows_i8_rounding_and_scale_range(dev, cols):
    """Bit-exact at the cases where a quotient computed other than by IEEE division would differ: exact ties
    (k + 0.5 at scale 1 and 0.5, rounding to even), scales on both sides of 2^-100 and 2^100 (the kernel switches its
    division method there), subnormal elements, and 1024 rows whose magnitudes run from 1e-38 to 1e38."""
    rng = np.random.default_rng(cols)
    rows = []
    ties = np.arange(-126.5, 127.0, 1.0, dtype=np.float32)              # every k + 0.5 in range
    row = np.resize(ties, cols).astype(np.float32)
    row[0] = 127.0                                                      # max 127: s = 1, quotients are exact ties
    rows.append(row)
    rows.append(row * np.float32(0.5))                                  # s = 0.5
    for e in (-101, -100, -99, 99, 100, 101):                          # s = mx / 127 around 2^-100 and 2^100
        for f in (0.999, 1.0, 1.001):
            r = (rng.standard_normal(cols) * 2.0 ** e).astype(np.float32)
            r[1] = np.float32(127 * f * 2.0 ** e)
            rows.append(r)
    r = (rng.standard_normal(cols) * 1e-39).astype(np.float32)          # every element subnormal
    rows.append(r)
    r = (rng.standard_normal(cols)).astype(np.float32)
    r[::7] = np.float32(1e-42)                                          # subnormals among normal values
    rows.append(r)
    mags = 10.0 ** rng.uniform(-38, 38, 1024 if cols <= 5120 else 64)
    rows += [(rng.standard_normal(cols) * m).astype(np.float32) for m in mags]
    w = np.stack(rows).astype(np.float32)
    assert np.isfinite(w).all()
    q, s = mh.quant_rows_i8(torch.from_numpy(w).to(dev))
    wq, ws = orc.quant_rows_i8(w)
    assert np.array_equal(s.cpu().numpy().view(np.uint32), ws.view(np.uint32))
    bad = np.argwhere(q.cpu().numpy() != wq)
    assert bad.size == 0, f"{len(bad)} differ, first at {bad[:3].tolist()}"


def fc1_inputs(rng, m, n, k):
    x = randn_bf16_bits(rng, (m, k))
    w = rng.integers(-127, 128, (2 * n, k), dtype=np.int8)
    s = rng.uniform(0.5e-3, 2e-3, 2 * n).astype(np.float32)
    return x, w, s


@pytest.mark.parametrize("m,n,k", [(1, 128, 64), (37, 128, 128), (256, 256, 512), (300, 384, 320), (513, 128, 5120)])
def test_gemm_w8a16_swiglu(dev, m, n, k):
    rng = np.random.default_rng(m + n + k)
    x, w, s = fc1_inputs(rng, m, n, k)
    want = orc.gemm_w8a16_swiglu(x, w, s)
    got = mh.gemm_w8a16_swiglu(from_bits(x, dev), torch.from_numpy(w).to(dev), torch.from_numpy(s).to(dev))
    g, wv = bits_to_f64(to_bits(got)), bits_to_f64(want)
    assert_close(g, wv, 1e-2, 1e-4, f"fc1 {m}x{n}x{k}")
    rel, cos = diff(g, wv, n)
    assert rel < 3e-3 and cos > 0.9999


def test_gemm_quantized_weights_end_to_end(dev):
    """quant_rows_i8 on bf16 weights, then the GEMM: equals the oracle run on the oracle's own quantization."""
    rng = np.random.default_rng(9)
    m, n, k = 100, 256, 1024
    x = randn_bf16_bits(rng, (m, k))
    wf = randn_bf16_bits(rng, (2 * n, k), 0.02)
    q, s = mh.quant_rows_i8(from_bits(wf, dev))
    got = mh.gemm_w8a16_swiglu(from_bits(x, dev), q, s)
    wq, ws = orc.quant_rows_i8(wf)
    want = orc.gemm_w8a16_swiglu(x, wq, ws)
    assert_close(bits_to_f64(to_bits(got)), bits_to_f64(want), 1e-2, 1e-6, "quantized fc1")


def test_gemm_768p_every_row(dev):
    """X bf16 [129,536 x 5120] ~ N(0,1), W int8 [27,648 x 5120] uniform in [-127,127], per-output-channel scales
    U(0.5e-3, 2e-3), into an output filled with NaN: every element against float64 products on the GPU over the same
    operands (so a tile left unwritten, or written twice from the wrong operands, fails), and 6 rows (both ends
    included) against the oracle over all 13,824 columns."""
    m, n, k = 129536, 13824, 5120
    gen = torch.Generator(device=dev).manual_seed(2)
    x = torch.randn((m, k), generator=gen, device=dev).to(torch.bfloat16)
    w = torch.randint(-127, 128, (2 * n, k), generator=gen, device=dev, dtype=torch.int8)
    s = (torch.rand(2 * n, generator=gen, device=dev) * 1.5e-3 + 0.5e-3).float()
    out = mh.gemm_w8a16_swiglu(x, w, s, out=nan_filled((m, n), dev))
    rel, cos = check_gemm_full(out, x, w, "fc1 W8A16 768p", w_scale=s, epi="swiglu")
    assert rel < 3e-3 and cos > 0.9999
    rows = np.array([0, 1, 255, 256, 77777, m - 1])
    ti = torch.from_numpy(rows).to(dev)
    want = orc.gemm_w8a16_swiglu(to_bits(x[ti]), w.cpu().numpy(), s.cpu().numpy())
    g = bits_to_f64(to_bits(out[ti]))
    assert_close(g, bits_to_f64(want), 1e-2, 1e-4, "fc1 768p")
    rel, cos = diff(g, bits_to_f64(want), n)
    assert rel < 3e-3 and cos > 0.9999


# ---- the dense bf16 fc1 (the --int8 none path) ----------------------------------------------------------------------

@pytest.mark.parametrize("m,n,k", [(1, 128, 64), (37, 128, 128), (300, 384, 320), (513, 128, 5120)])
def test_gemm_bf16_swiglu(dev, m, n, k):
    rng = np.random.default_rng(m * 3 + n + k)
    x = randn_bf16_bits(rng, (m, k))
    w = randn_bf16_bits(rng, (2 * n, k), 0.05)
    want = orc.gemm_bf16_swiglu(x, w)
    got = mh.gemm_bf16_swiglu(from_bits(x, dev), from_bits(w, dev))
    g, wv = bits_to_f64(to_bits(got)), bits_to_f64(want)
    assert_close(g, wv, 1e-2, 1e-4, f"bf16 fc1 {m}x{n}x{k}")
    rel, cos = diff(g, wv, n)
    assert rel < 3e-3 and cos > 0.9999


def test_gemm_bf16_equals_int8_path_on_integer_weights(dev):
    """Integer weights |w| <= 127 are exact in bf16 and int8, so with unit scales both paths compute the same sums
    in the same order: identical outputs."""
    rng = np.random.default_rng(21)
    m, n, k = 300, 256, 640
    x = randn_bf16_bits(rng, (m, k))
    wi = rng.integers(-127, 128, (2 * n, k), dtype=np.int8)
    tw8 = torch.from_numpy(wi).to(dev)
    ones = torch.ones(2 * n, dtype=torch.float32, device=dev)
    a = mh.gemm_w8a16_swiglu(from_bits(x, dev), tw8, ones)
    b = mh.gemm_bf16_swiglu(from_bits(x, dev), tw8.to(torch.bfloat16))
    assert torch.equal(a.view(torch.int16), b.view(torch.int16))


def test_gemm_bf16_768p_every_row(dev):
    """X bf16 [129,536 x 5120] ~ N(0,1), W bf16 [27,648 x 5120] ~ N(0, 0.02), into a NaN-filled output: every
    element against float64 products on the GPU; 6 rows against the oracle over all 13,824 columns."""
    m, n, k = 129536, 13824, 5120
    gen = torch.Generator(device=dev).manual_seed(4)
    x = torch.randn((m, k), generator=gen, device=dev).to(torch.bfloat16)
    w = (0.02 * torch.randn((2 * n, k), generator=gen, device=dev)).to(torch.bfloat16)
    out = mh.gemm_bf16_swiglu(x, w, out=nan_filled((m, n), dev))
    rel, cos = check_gemm_full(out, x, w, "fc1 bf16 768p", epi="swiglu")
    assert rel < 3e-3 and cos > 0.9999
    rows = np.array([0, 1, 255, 256, 77777, m - 1])
    ti = torch.from_numpy(rows).to(dev)
    want = orc.gemm_bf16_swiglu(to_bits(x[ti]), to_bits(w))
    g = bits_to_f64(to_bits(out[ti]))
    assert_close(g, bits_to_f64(want), 1e-2, 1e-4, "bf16 fc1 768p")
    rel, cos = diff(g, bits_to_f64(want), n)
    assert rel < 3e-3 and cos > 0.9999


# ---- the reference's W8A8 fc1 (int8 activations and weights, int8 MFMA) ------------------------------------------

@pytest.mark.parametrize("m,n,k", [(1, 128, 128), (37, 128, 256), (300, 384, 384), (513, 128, 5120)])
def test_gemm_i8_swiglu(dev, m, n, k):
    rng = np.random.default_rng(m * 5 + n + k)
    x = rng.integers(-127, 128, (m, k), dtype=np.int8)
    w = rng.integers(-127, 128, (2 * n, k), dtype=np.int8)
    sx = rng.uniform(0.005, 0.05, m).astype(np.float32)
    sw = rng.uniform(0.5e-3, 2e-3, 2 * n).astype(np.float32)
    want = orc.gemm_i8_swiglu(x, sx, w, sw)
    t = lambda a: torch.from_numpy(a).to(dev)  # noqa: E731
    got = mh.gemm_i8_swiglu(t(x), t(sx), t(w), t(sw))
    g, wv = bits_to_f64(to_bits(got)), bits_to_f64(want)
    assert_close(g, wv, 1e-2, 1e-4, f"int8 fc1 {m}x{n}x{k}")
    rel, cos = diff(g, wv, n)
    assert rel < 3e-3 and cos > 0.9999


def test_gemm_i8_quantized_activations_end_to_end(dev):
    """quant_rows_i8 of bf16 x and of bf16 weights, then the W8A8 GEMM: equals the oracle on the oracle's own
    quantizations (bit-exact inputs), and stays within the int8 error budget of the bf16 fc1."""
    rng = np.random.default_rng(22)
    m, n, k = 200, 256, 1024
    x = randn_bf16_bits(rng, (m, k))
    wf = randn_bf16_bits(rng, (2 * n, k), 0.02)
    xq, xs = mh.quant_rows_i8(from_bits(x, dev))
    wq, ws = mh.quant_rows_i8(from_bits(wf, dev))
    got = mh.gemm_i8_swiglu(xq, xs, wq, ws)
    oxq, oxs = orc.quant_rows_i8(x)
    owq, ows = orc.quant_rows_i8(wf)
    want = orc.gemm_i8_swiglu(oxq, oxs, owq, ows)
    assert_close(bits_to_f64(to_bits(got)), bits_to_f64(want), 1e-2, 1e-6, "W8A8 fc1")
    dense = bits_to_f64(orc.gemm_bf16_swiglu(x, wf))
    rel, _ = diff(bits_to_f64(to_bits(got)), dense, n)
    assert rel < 0.1, rel  # the reference reports a few 1e-2 for int8 fc1 + fc2 (docs/performance.md:147-152)


def test_gemm_i8_768p_every_row(dev):
    """The W8A8 fc1 at 768p into a NaN-filled output: every element against float64 products of the int8 operands and
    both scales on the GPU; 6 rows against the oracle."""
    m, n, k = 129536, 13824, 5120
    gen = torch.Generator(device=dev).manual_seed(6)
    x = torch.randint(-127, 128, (m, k), generator=gen, device=dev, dtype=torch.int8)
    w = torch.randint(-127, 128, (2 * n, k), generator=gen, device=dev, dtype=torch.int8)
    sx = (torch.rand(m, generator=gen, device=dev) * 0.01 + 0.005).float()
    sw = (torch.rand(2 * n, generator=gen, device=dev) * 1.5e-3 + 0.5e-3).float()
    out = mh.gemm_i8_swiglu(x, sx, w, sw, out=nan_filled((m, n), dev))
    rel, cos = check_gemm_full(out, x, w, "fc1 W8A8 768p", x_scale=sx, w_scale=sw, epi="swiglu")
    assert rel < 3e-3 and cos > 0.9999
    rows = np.array([0, 1, 255, 256, 77777, m - 1])
    ti = torch.from_numpy(rows).to(dev)
    want = orc.gemm_i8_swiglu(x[ti].cpu().numpy(), sx[ti].cpu().numpy(), w.cpu().numpy(), sw.cpu().numpy())
    g = bits_to_f64(to_bits(out[ti]))
    assert_close(g, bits_to_f64(want), 1e-2, 1e-4, "int8 fc1 768p")


def chosen_tile(m, nt, cus=256):
    """The rows and columns of the tile that a launch of m rows and nt column tiles takes: the rule of choose_tile over
    the table in the kernels' source."""
    src = (Path(__file__).resolve().parent.parent / "mako-video_amd" / "csrc" / "gemm.hip").read_text()
    table = re.search(r"kTiles\[\] = \{(.*?)\};", src)[1]
    tiles = [tuple(map(int, t.split(","))) for t in re.findall(r"\{([^}]*)\}", table)]
    return min(tiles, key=lambda t: -(-(-(-m // t[0]) * nt * (128 // t[1])) // cus) * t[2])[:2]


@pytest.mark.parametrize("form,k", [(form, k) for form in ("w8a16", "bf16", "w8a8")
                                    for k in (64, 128, 192, 256, 320, 384, 640) if form != "w8a8" or k % 128 == 0])
def test_gemm_row_tiles(dev, form, k):
    """Every tile (64 column tiles on 256 CUs: 1021 rows take 256-row tiles, 763 192, 505 128, 255 64, 33 the narrow
    one, by the launch's own table of costs), its last rows missing, at K-step counts around the LDS rings' depths: every element against float64 products, and the
    rows of a smaller batch bit-identical to the same rows of the larger one (the row tile changes no sum's order)."""
    assert torch.cuda.get_device_properties(dev).multi_processor_count == 256
    assert [chosen_tile(m, 64) for m in (1021, 763, 505, 255, 33)] == [(256, 128), (192, 128), (128, 128), (64, 128),
                                                                     (64, 32)]
    g = torch.Generator(device=dev).manual_seed(k)
    m_max, n = 1021, 64 * 128
    xf = torch.randn((m_max, k), generator=g, device=dev).to(torch.bfloat16)
    wf = (0.02 * torch.randn((2 * n, k), generator=g, device=dev)).to(torch.bfloat16)
    x, xs = mh.quant_rows_i8(xf) if form == "w8a8" else (xf, None)
    w, ws = (wf, None) if form == "bf16" else mh.quant_rows_i8(wf)
    gate = torch.randn(2 * n, generator=g, device=dev)
    res0 = torch.randn((m_max, 2 * n), generator=g, device=dev)

    def run(m):
        xm, sm = x[:m], None if xs is None else xs[:m].contiguous()
        if form == "w8a16":
            f = mh.gemm_w8a16_swiglu(xm, w, ws, out=nan_filled((m, n), dev))
        elif form == "bf16":
            f = mh.gemm_bf16_swiglu(xm, w, out=nan_filled((m, n), dev))
        else:
            f = mh.gemm_i8_swiglu(xm, sm, w, ws, out=nan_filled((m, n), dev))
        y = mh.gemm(xm, w, x_scale=sm, w_scale=ws, out=nan_filled((m, 2 * n), dev))
        r = mh.gemm_gate_add(xm, w, res0[:m].to(torch.bfloat16), gate, x_scale=sm, w_scale=ws)
        r32 = mh.gemm_gate_add(xm, w, res0[:m].clone(), gate, x_scale=sm, w_scale=ws)
        return f, y, r, r32

    full = run(m_max)
    check_gemm_full(full[0], x, w, f"{form} fc1", x_scale=xs, w_scale=ws, epi="swiglu")
    check_gemm_full(full[1], x, w, f"{form} store", x_scale=xs, w_scale=ws)
    check_gemm_full(full[2], x, w, f"{form} gate_add", x_scale=xs, w_scale=ws, epi="gate_add",
                    residual0=res0.to(torch.bfloat16), gate=gate)
    check_gemm_full(full[3], x, w, f"{form} gate_add_f32", x_scale=xs, w_scale=ws, epi="gate_add", residual0=res0,
                    gate=gate)
    for m in (763, 505, 255, 33):
        for name, a, b in zip(("fc1", "store", "gate_add", "gate_add_f32"), run(m), full):
            assert torch.equal(a, b[:m]), f"{form} {name} k {k} m {m}"


@pytest.mark.parametrize("form", ["w8a16", "bf16"])
@pytest.mark.parametrize("steps", [1, 2, 3, 4, 5, 6, 7, 8, 9, 10, 11, 13])
def test_gemm_narrow_k_steps(dev, form, steps):
    """The narrow tile (33 rows of 64 column tiles on 256 CUs) at every K-step count around its rings' depth and its
    loop's three steps: every element against float64 products, and bit-identical to a larger tile's."""
    k, n = 64 * steps, 64 * 128
    g = torch.Generator(device=dev).manual_seed(steps)
    x = torch.randn((1021, k), generator=g, device=dev).to(torch.bfloat16)
    wf = (0.02 * torch.randn((2 * n, k), generator=g, device=dev)).to(torch.bfloat16)
    w, ws = (wf, None) if form == "bf16" else mh.quant_rows_i8(wf)
    y = mh.gemm(x[:33], w, w_scale=ws, out=nan_filled((33, 2 * n), dev))
    check_gemm_full(y, x[:33], w, f"{form} k {k}", w_scale=ws)
    assert torch.equal(y, mh.gemm(x, w, w_scale=ws, out=nan_filled((1021, 2 * n), dev))[:33])
