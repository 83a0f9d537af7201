"""Parity of the HIP GEMM / quantisation kernels with the CPU oracle (GPU).

Bars: int8 and fp8 codes and scales bit-exact; int8 int32 accumulators bit-exact; bf16
outputs within two bf16 rounding steps of the fp32/float64 oracle (different fp32
summation order); fp8 GEMM within 2e-2 max-abs and cosine >= 0.9995 of the dequantised
float64 product.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import branch_oracle as bo
from oracle import quant_oracle as qo

pytestmark = pytest.mark.gpu


def _rand(shape, seed, scale=1.0, dtype=torch.bfloat16):
    g = torch.Generator().manual_seed(seed)
    return (torch.randn(shape, generator=g) * scale).to(dtype)


def assert_bf16_close(got, want, steps=2, atol=1e-6):
    got, want = got.float().cpu(), want.float().cpu()
    tol = steps * 2.0 ** -8 * want.abs() + atol
    bad = (got - want).abs() > tol
    assert not bool(bad.any()), f"{int(bad.sum())} values off; max err {(got - want).abs().max().item():.3e}"


@pytest.mark.parametrize("m,n,k", [(300, 200, 192), (128, 128, 64), (37, 5120, 128), (1000, 40, 5120)])
def test_bf16_linear(device, m, n, k):
    from vdn_h3_amd import linear

    print(f"case bf16 linear {m}x{n}x{k}", flush=True)
    x, w = _rand((m, k), 1), _rand((n, k), 2, 0.05)
    got = linear.linear(x.to(device), w.to(device))
    torch.cuda.synchronize()
    assert_bf16_close(got, (x.double() @ w.double().t()).to(torch.bfloat16))


def test_sigmoid_bias_and_accumulate_epilogues(device):
    from vdn_h3_amd import linear

    print("case epilogues", flush=True)
    m, n, k = 257, 130, 256
    x, w = _rand((m, k), 3), _rand((n, k), 4, 0.05)
    b = _rand((n,), 5, 0.5)
    got = linear.sigmoid_linear(x.to(device), w.to(device), b.to(device))
    want = torch.sigmoid(bo.linear_bf16(x, w, b))
    # a pre-activation one bf16 step away (fp32 summation order) moves the sigmoid by <= 2^-8
    assert_bf16_close(got, want, steps=2, atol=2.0 ** -8)
    base = _rand((m, n), 6)
    out = base.to(device)
    linear.linear(x.to(device), w.to(device), out=out, accumulate=True)
    torch.cuda.synchronize()
    want = (base.float() + bo.linear_bf16(x, w).float()).to(torch.bfloat16)
    assert_bf16_close(out, want, steps=2)


def test_split_sigmoid_epilogue_equals_two_gemms(device):
    """beta and the output-gate down-projection as one GEMM (sigmoid on the first 40 columns only)
    equal sigmoid_linear and linear run separately, bit for bit."""
    from vdn_h3_amd import linear as L

    m, k, heads, rank = 1000, 5120, 40, 128
    x = _rand((m, k), 21).to(device)
    wb, wd = _rand((heads, k), 22, 0.02).to(device), _rand((rank, k), 23, 0.02).to(device)
    both = L.sigmoid_linear_split(x, torch.cat([wb, wd]).contiguous(), heads)
    torch.cuda.synchronize()
    assert torch.equal(both[:, :heads], L.sigmoid_linear(x, wb))
    assert torch.equal(both[:, heads:], L.linear(x, wd))
    with pytest.raises(ValueError):
        L.gemm(L.KIND_BF16, x, wb, act="sigmoid", act_cols=heads + 1)


@pytest.mark.parametrize("m,k", [(257, 512), (64, 5120), (33, 1032), (5, 2048), (5, 2056), (5, 5128),
                                 (9, 8192), (7, 8200)])
def test_quant_codes_bit_exact(device, m, k):
    from vdn_h3_amd import linear

    print(f"case quant codes {m}x{k}", flush=True)
    x = _rand((m, k), 8, 3.0)
    x[3] = 0.0
    q8, s8 = linear.quantize_rows(x.to(device), linear.KIND_I8)
    wq8, ws8 = qo.int8_quantize_rows(x)
    assert torch.equal(q8.cpu(), wq8) and torch.equal(s8.cpu(), ws8)
    qf, sf = linear.quantize_rows(x.to(device), linear.KIND_F8)
    wqf, wsf = qo.fp8_quantize_rows(x)
    assert torch.equal(qf.cpu().view(torch.uint8), wqf.view(torch.uint8)) and torch.equal(sf.cpu(), wsf)
    qt, st = linear.quantize_tensor_fp8(x.to(device))
    wqt, wst = qo.fp8_quantize_tensor(x)
    assert torch.equal(qt.cpu().view(torch.uint8), wqt.view(torch.uint8)) and torch.equal(st.cpu(), wst)


def test_fp8_encoder_covers_every_bf16_magnitude(device):
    """Every finite bf16 value below 448, quantised with scale 1, matches torch's e4m3fn cast."""
    from vdn_h3_amd import linear

    print("case fp8 exhaustive", flush=True)
    bits = torch.arange(0, 1 << 16, dtype=torch.int32).to(torch.int16).view(torch.bfloat16)
    vals = bits.float()
    keep = torch.isfinite(vals) & (vals.abs() <= 448.0)
    vals = vals[keep]
    n = (vals.numel() // 8) * 8
    row = torch.cat([vals[:n], torch.tensor([448.0] * 8)]).to(torch.bfloat16).reshape(1, -1)
    q, s = linear.quantize_rows(row.to(device), linear.KIND_F8)
    assert s.item() == 1.0
    want = row.float().clamp(-448, 448).to(torch.float8_e4m3fn).view(torch.uint8)
    assert torch.equal(q.cpu().view(torch.uint8), want)


@pytest.mark.parametrize("m,n,k", [(300, 200, 256), (129, 257, 1024)])
def test_int8_accumulators_bit_exact_and_scaled_output(device, m, n, k):
    from vdn_h3_amd import linear

    print(f"case int8 {m}x{n}x{k}", flush=True)
    x, w = _rand((m, k), 9), _rand((n, k), 10, 0.02)
    xq, xs = qo.int8_quantize_rows(x)
    wq, ws = qo.int8_quantize_rows(w)
    acc = linear.int8_accumulators(xq.to(device), wq.to(device))
    assert torch.equal(acc.cpu(), qo.int8_accumulate(xq, wq))
    out = linear.gemm_w8a8(xq.to(device), xs.to(device), wq.to(device), ws.to(device))
    assert_bf16_close(out, qo.int8_linear(xq, xs, wq, ws), steps=1)


@pytest.mark.parametrize("per_tensor", [False, True])
def test_fp8_gemm(device, per_tensor):
    from vdn_h3_amd import fp8

    print(f"case fp8 gemm per_tensor={per_tensor}", flush=True)
    m, n, k = 333, 256, 640
    x, w = _rand((m, k), 11), _rand((n, k), 12, 0.02)
    xq, xs = fp8.quantize_activation(x.to(device), per_tensor=per_tensor)
    wq, ws = fp8.quantize_weight(w.to(device), per_tensor=per_tensor)
    got = fp8.project(x.to(device), {fp8.FP8_WEIGHT_KEY: wq, fp8.FP8_SCALE_KEY: ws}).float().cpu()
    want = qo.fp8_linear(xq.cpu(), xs.cpu(), wq.cpu(), ws.cpu()).float()
    err = (got - want).abs().max().item()
    cos = torch.nn.functional.cosine_similarity(got.double().flatten(), want.double().flatten(), dim=0).item()
    assert err <= 2e-2 and cos >= 0.9995, (err, cos)


def test_projection_dispatch(device):
    from vdn_h3_amd import projection

    print("case projection dispatch", flush=True)
    x, w = _rand((200, 256), 13), _rand((128, 256), 14, 0.02)
    bf = projection.project(x.to(device), {"to_out_linear.weight": w.to(device)})
    assert_bf16_close(bf, bo.linear_bf16(x, w))
    maps, info = projection.prepare_int8_projection_maps([{"to_out_linear.weight": w}], device)
    assert info.quantized_blocks == 1 and maps[0]["to_out_linear.weight_fp8"].dtype == torch.int8
    got = projection.project(x.to(device), maps[0])
    xq, xs = qo.int8_quantize_rows(x)
    wq, ws = qo.int8_quantize_rows(w)
    assert_bf16_close(got, qo.int8_linear(xq, xs, wq, ws), steps=1)


def test_full_shape_int8_qkv_accumulators_sampled(device):
    """M=40,688, K=5,120, N=15,360 W8A8 int8: all accumulators on the GPU, sampled rows checked exactly."""
    from vdn_h3_amd import linear, synth

    print("case full-shape int8 qkv", flush=True)
    m, k, n = 40688, 5120, 15360
    x = synth.randn((m, k), 30, device=device, dtype=torch.bfloat16)
    w = synth.randn((n, k), 31, device=device, dtype=torch.bfloat16, scale=0.02)
    xq, xs = linear.quantize_rows(x, linear.KIND_I8)
    wq, ws = linear.quantize_rows(w, linear.KIND_I8)
    acc = linear.int8_accumulators(xq, wq)
    torch.cuda.synchronize()
    # one row of every 256-row M tile plus the tiles' edge rows; the int32 sums are formed in float64, where
    # they are exact (every product is at most 127^2, a row of 5120 of them sums to < 2^27)
    rows = torch.tensor(sorted(set(_tile_rows(m).tolist() + [0, 1, 127, 128, 255, 256, 40573, 40687])))
    a = xq[rows.to(device)].cpu()
    want = (a.double() @ wq.cpu().double().T).to(torch.int32)
    print(f"  {len(rows)} rows checked", flush=True)
    assert torch.equal(acc[rows.to(device)].cpu(), want)
    assert torch.equal(xq.cpu()[rows], qo.int8_quantize_rows(x.cpu()[rows])[0])


def _tile_rows(m, tile=256):
    """One row per 256-row M tile, at a position that walks through the tile, plus the last row."""
    rows = [t + (37 * i) % min(tile, m - t) for i, t in enumerate(range(0, m, tile))]
    return torch.tensor(sorted(set(rows + [m - 1])))


@pytest.mark.parametrize("n", [15360, 5120])
def test_full_shape_fp8_per_tensor_sampled(device, n):
    """M=40,688, K=5,120 fp8 e4m3 with per-tensor scales (the reference's fp8 W8A8 variant), N=15,360
    (qkv) and 5,120 (out): one row of every M tile against the dequantised float64 product."""
    from vdn_h3_amd import fp8, synth

    print(f"case full-shape fp8 per-tensor N={n}", flush=True)
    m, k = 40688, 5120
    x = synth.randn((m, k), 32, device=device, dtype=torch.bfloat16)
    w = synth.randn((n, k), 33, device=device, dtype=torch.bfloat16, scale=0.02)
    xq, xs = fp8.quantize_activation(x, per_tensor=True)
    wq, ws = fp8.quantize_weight(w, per_tensor=True)
    got = fp8.project(x, {fp8.FP8_WEIGHT_KEY: wq, fp8.FP8_SCALE_KEY: ws})
    torch.cuda.synchronize()
    rows = _tile_rows(m)
    want = qo.fp8_linear(xq[rows.to(device)].cpu(), xs.cpu(), wq.cpu(), ws.cpu()).float()
    g = got[rows.to(device)].float().cpu()
    err = (g - want).abs().max().item()
    cos = torch.nn.functional.cosine_similarity(g.double().flatten(), want.double().flatten(), dim=0).item()
    print(f"  {len(rows)} rows: max abs {err:.3e}, cosine {cos:.7f}", flush=True)
    # outputs reach |7| (K = 5120 products of N(0,1) x N(0, 0.02^2)), where one bf16 step is 2^-5: the bar
    # is one rounding step of the float64 product (fp32 accumulation order), and max-abs 2e-2 where |want| < 2
    assert cos >= 0.9995, cos
    # per value: one bf16 ulp of the float64 product, plus 2^-12 for the fp32 accumulation of 5120 products
    # (outputs near zero carry that absolute noise, many of their own ulps)
    ulp = torch.ldexp(torch.ones_like(want), torch.frexp(want)[1] - 8).clamp_min(2.0 ** -133)
    excess = ((g - want).abs() - 2.0 ** -12).clamp_min(0) / ulp
    print(f"  beyond 2^-12, in ulps of the float64 value: max {excess.max().item():.2f}", flush=True)
    assert excess.max().item() <= 1.0
    assert (g - want).abs()[want.abs() < 2].max().item() <= 2e-2


def test_full_shape_int8_out_projection_sampled(device):
    """The out-projection shape M=40,688, K=5,120, N=5,120 W8A8 int8: the int32 accumulators of one row
    per M tile bit-exact, and the scaled bf16 output within one rounding step."""
    from vdn_h3_amd import linear, synth

    print("case full-shape int8 out", flush=True)
    m, k, n = 40688, 5120, 5120
    x = synth.randn((m, k), 34, device=device, dtype=torch.bfloat16)
    w = synth.randn((n, k), 35, device=device, dtype=torch.bfloat16, scale=0.02)
    xq, xs = linear.quantize_rows(x, linear.KIND_I8)
    wq, ws = linear.quantize_rows(w, linear.KIND_I8)
    acc = linear.int8_accumulators(xq, wq)
    out = linear.gemm_w8a8(xq, xs, wq, ws.reshape(1, -1))
    torch.cuda.synchronize()
    rows = _tile_rows(m)
    a = xq[rows.to(device)].cpu().numpy().astype(np.int64)
    b = wq.cpu().numpy().astype(np.int64)
    want_acc = torch.from_numpy((a @ b.T).astype(np.int32))
    assert torch.equal(acc[rows.to(device)].cpu(), want_acc)
    want = qo.int8_linear(xq[rows.to(device)].cpu(), xs[rows.to(device)].cpu(), wq.cpu(), ws.cpu().reshape(1, -1))
    assert_bf16_close(out[rows.to(device)], want, steps=1)


# sizes of every tile height the launcher can pick (32 mi rows: the fewest rounds over 256 CUs), each with a ragged
# last tile row, N a multiple of 8, of 4 and odd (whole and partly stored last columns), and 1 to 5 stages of 128 K
# bytes
TILE_SIZES = [(1, 8), (31, 20), (65, 257), (511, 15100), (1000, 5113), (513, 15100), (1801, 5113), (2303, 5116),
              (2561, 5120), (2881, 4900), (4100, 5128)]


def test_tile_sizes_cover_every_height():
    from vdn_h3_amd import _lib

    heights = {_lib.lib().vdnh3_gemm_tile_rows(m, n) for m, n in TILE_SIZES}
    assert heights == {32 * mi for mi in (2, 4, 5, 6, 7, 8)}


@pytest.mark.parametrize("stages", [1, 2, 3, 5])
@pytest.mark.parametrize("m,n", TILE_SIZES)
def test_tile_heights_widths_and_stages(device, m, n, stages):
    from vdn_h3_amd import linear

    print(f"case tiles {m}x{n}, {stages} stages", flush=True)
    # int8: exact integers; the bf16 output rounds acc * a_scale * b_scale once
    k = 128 * stages
    g = torch.Generator(device="cuda").manual_seed(m * 7 + n + stages)
    aq = torch.randint(-127, 128, (m, k), generator=g, device=device, dtype=torch.int8)
    bq = torch.randint(-127, 128, (n, k), generator=g, device=device, dtype=torch.int8)
    a_s = torch.rand(m, 1, generator=g, device=device) * 1e-2
    b_s = torch.rand(1, n, generator=g, device=device) * 1e-2
    acc = (aq.float() @ bq.float().t())  # at most 640 products below 2^14: exact in fp32
    assert torch.equal(linear.int8_accumulators(aq, bq), acc.to(torch.int32))
    assert torch.equal(linear.gemm_w8a8(aq, a_s, bq, b_s), (acc * a_s * b_s).to(torch.bfloat16))
    assert torch.equal(linear.gemm_w8a8(aq, a_s, bq, b_s, out_dtype=torch.float32), acc * a_s * b_s)
    # bf16: fp32 sums of K products; fp8: the instruction keeps about 15 bits below the largest products it sums
    # (measured: at most 2^-15 of sum |a b| off the exact sum, in its 32x32 and 16x16 shapes alike). Then one
    # rounding (2^-9 relative; 2^-8 leaves room for a tie).
    for kind in ("fp8", "bf16"):
        k = (128 if kind == "fp8" else 64) * stages
        a = torch.randn(m, k, generator=g, device=device).to(torch.bfloat16)
        b = (torch.randn(n, k, generator=g, device=device) * 0.1).to(torch.bfloat16)
        base = torch.randn(m, n, generator=g, device=device).to(torch.bfloat16)
        out = base.clone()
        if kind == "fp8":
            a, b = a.to(torch.float8_e4m3fn), b.to(torch.float8_e4m3fn)
            one = torch.ones(1, 1, device=device)
            got = linear.gemm_w8a8(a, one, b, one)
            linear.gemm_w8a8(a, one, b, one, out=out, accumulate=True)
        else:
            got = linear.linear(a, b)
            linear.linear(a, b, out=out, accumulate=True)
        ad, bd = a.double(), b.double()
        want = ad @ bd.t()
        bound = (2.0 ** -14 if kind == "fp8" else k * 2.0 ** -24) * (ad.abs() @ bd.abs().t())
        assert bool(((got.double() - want).abs() <= bound + 2.0 ** -8 * want.abs()).all()), kind
        assert torch.equal(out, (base.float() + got.float()).to(torch.bfloat16)), kind


@pytest.mark.parametrize("m,n", TILE_SIZES)
def test_32_bit_outputs_any_alignment(device, m, n):
    """fp32 and int32 outputs, written and accumulated, into rows of any 4-byte alignment; the rest of them untouched."""
    from vdn_h3_amd import linear

    print(f"case 32-bit outputs {m}x{n}", flush=True)
    k = 256
    g = torch.Generator(device="cuda").manual_seed(m + 3 * n)
    a = torch.randint(-127, 128, (m, k), generator=g, device=device, dtype=torch.int8)
    b = torch.randint(-127, 128, (n, k), generator=g, device=device, dtype=torch.int8)
    a_s = torch.rand(m, 1, generator=g, device=device) * 1e-2
    b_s = torch.rand(1, n, generator=g, device=device) * 1e-2
    acc = a.float() @ b.float().t()  # at most 256 products below 2^14: exact in fp32
    base = torch.randn(m, n + 3, generator=g, device=device)
    for first in (0, 1, 2, 3):
        for accumulate in (False, True):
            whole = base.clone()
            out = whole[:, first:first + n]
            linear.gemm_w8a8(a, a_s, b, b_s, out=out, out_dtype=torch.float32, accumulate=accumulate)
            want = base.clone()
            want[:, first:first + n] = acc * a_s * b_s + (base[:, first:first + n] if accumulate else 0)
            assert torch.equal(whole, want), (first, accumulate)
        ints = torch.full((m, n + 3), 7, dtype=torch.int32, device=device)
        linear.gemm(linear.KIND_I8, a, b, out=ints[:, first:first + n], out_dtype=torch.int32)
        want = torch.full_like(ints, 7)
        want[:, first:first + n] = acc.to(torch.int32)
        assert torch.equal(ints, want), first


@pytest.mark.parametrize("kind,dtype,k,per_lane", [
    (0, torch.bfloat16, 16, 2), (1, torch.int8, 32, 2), (2, torch.float8_e4m3fn, 64, 2),        # 4 accumulators of 16
    (3, torch.bfloat16, 32, 2), (4, torch.int8, 64, 2), (5, torch.float8_e4m3fn, 128, 1)])     # 32 accumulators of 4
def test_mfma_rate_kernels_do_their_products(device, kind, dtype, k, per_lane):
    """Operands of ones: a lane's checksum counts the products of its MFMAs (``per_lane`` on each accumulator a pass)."""
    from vdn_h3_amd import _lib

    iters, blocks = 3, 4
    ones = torch.ones(8 * 64 * 32 // dtype.itemsize, dtype=torch.float32).to(dtype).to(device)
    out = torch.empty(blocks * 256, dtype=torch.float32, device=device)
    lib = _lib.lib()
    _lib.check(lib.vdnh3_mfma_peak(kind, _lib.ptr(ones), _lib.ptr(ones), iters, blocks, _lib.ptr(out),
                                   _lib.stream_handle(device)), "mfma_peak")
    values = 4 * 16 if kind < 3 else 32 * 4
    assert bool((out == values * per_lane * iters * k).all())
    assert lib.vdnh3_mfma_peak_ops(kind, iters, blocks) == 2 * values * 64 * per_lane * iters * k * 4 * blocks
