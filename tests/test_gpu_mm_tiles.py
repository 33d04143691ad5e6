"""The kernels of the linear-layer product (mm_skinny, mm_ksplit, mm_bf16)
against the float64 product of the same BF16-rounded operands: tokens at and
past every boundary of the kernel choice and of the tiles, outputs that end
inside a tile, k of one half stage, whole stages, a half last one and more
stages than the LDS rings hold, rows with padding behind them."""
import ctypes

import numpy as np
import pytest
import torch

import kd_mm
import kd_oracle_quant as oq

pytestmark = pytest.mark.gpu

DEV = "cuda:0"

# M, N, K (test_mm_plan.py holds the kernel and tile that each takes)
CASES = [(1, 4, 32), (8, 36, 96), (9, 100, 416), (16, 260, 1184), (3, 16388, 288), (12, 16384, 64),
         (17, 32, 64), (33, 100, 544),
         (31, 8200, 160),     # 64 x 32
         (130, 4100, 96),     # 64 x 64
         (300, 4096, 416),    # 64 x 96
         (850, 2100, 672),    # 128 x 64
         (700, 4100, 352),    # 128 x 128
         (1030, 8000, 736),   # 128 x 96
         (1540, 4100, 96), (1700, 4096, 32), (2047, 4004, 352),   # 256 x 128
         (3900, 4080, 96), (3841, 4064, 64), (4090, 4064, 416)]   # 256 x 256
# k of several times the stages that the LDS rings hold: every buffer is
# refilled after it has been read, and the steady loops run; an odd and an
# even number of 64-k stages, whole and with a half last one
DEEP = [(M, N, K) for M, N, ks in [
    (2, 260, (2816, 2848, 2880)), (12, 260, (2816, 2848, 2880)), (2, 16388, (2848, 2880)), (12, 16388, (2848, 2880)),
    (33, 112, (832, 864, 896, 928)),      # 32 x 32
    (34, 4144, (832, 864, 896, 928)),     # 64 x 32
    (99, 4184, (832, 864, 896, 928)),     # 64 x 64
    (3347, 260, (832, 864, 896, 928)),    # 64 x 96
    (291, 4148, (832, 864, 928)),         # 128 x 64
    (3274, 524, (832, 864, 928)),         # 128 x 96
    (4048, 648, (832, 864, 928)),         # 128 x 128
    (3601, 1044, (832, 864)),             # 256 x 128
    (4057, 2180, (832, 864))] for K in ks]   # 256 x 256
# the large tiles' last steps, apart from their loop, with every number of
# stages up to those that the loop begins with: 256 x 256, 256 x 128
ENDS = [(M, N, K) for M, N in ((33001, 132), (1540, 4100)) for K in range(32, 321, 32)]


@pytest.mark.parametrize("xdt", [torch.float32, torch.bfloat16], ids=["f32", "bf16"])
@pytest.mark.parametrize("case", CASES + DEEP + ENDS, ids=lambda c: "x".join(map(str, c)))
def test_every_tile(case, xdt):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    M, N, K = case
    print(f"[case] mm {case} {xdt}", flush=True)
    g = torch.Generator().manual_seed(M + N + K)
    # rows of a wider matrix: what lies behind a row is never part of it
    w = torch.full((N, K + 8), float("nan"), dtype=torch.bfloat16)
    w[:, :K] = torch.randn((N, K), generator=g) * 0.05
    x = torch.full((M, K + 8), float("nan"), dtype=xdt)
    x[:, :K] = torch.randn((M, K), generator=g)
    bias = torch.randn(N, generator=g) * 0.1 if N % 8 else None
    out = torch.full((M + 1, N + 4), 7.0, device=DEV)
    d = kd_mm.make_desc(w.to(DEV)[:, :K], x.to(DEV)[:, :K], None if bias is None else bias.to(DEV), out[:M, :N])
    assert kd_mm.run_desc(d) == 0
    torch.cuda.synchronize()
    wr = w[:, :K].double()
    xr = torch.from_numpy(oq.round_bf16(x[:, :K].float().numpy())).double()
    ref = xr @ wr.T + (0.0 if bias is None else bias.double())
    # F32 accumulation of K products in any order: K rounding errors of 2^-24 of the sum of magnitudes at most
    limit = (xr.abs() @ wr.abs().T + (0.0 if bias is None else bias.double().abs())) * (K + 8) * 2.0 ** -24 + 1e-30
    got = out.cpu()
    err = (got[:M, :N].double() - ref).abs()
    assert bool((err <= limit).all()), float((err / limit).max())
    assert bool((got[M:] == 7.0).all()) and bool((got[:, N:] == 7.0).all())
    assert kd_mm.run_desc(d) == 0
    torch.cuda.synchronize()
    assert np.array_equal(out.cpu().numpy(), got.numpy())


@pytest.mark.parametrize("case", [(2, 260, 2848), (33, 112, 864), (99, 4184, 96), (300, 4096, 416), (1540, 4100, 96),
                                  (4057, 2180, 832)], ids=lambda c: "x".join(map(str, c)))
def test_f32_x_has_the_bits_of_its_rounding(case):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    M, N, K = case
    print(f"[case] mm x types {case}", flush=True)
    g = torch.Generator().manual_seed(M + N + K)
    w = (torch.randn((N, K), generator=g) * 0.05).bfloat16().to(DEV)
    x = torch.randn((M, K), generator=g).to(DEV)
    outs = [kd_mm.linear(v, w) for v in (x, x.bfloat16())]
    torch.cuda.synchronize()
    assert torch.equal(*outs)


@pytest.mark.parametrize("shape", [(1, 32), (3, 96), (71, 352), (129, 4096)], ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("kind", ["q8_0", "q4_0", "bf16", "f16", "f32"])
def test_dequant_padded_rows(kind, shape):
    """Rows back to back and rows with padding behind them: bitwise the
    oracle's values rounded to BF16, up to the last row and no further."""
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    N, K = shape
    print(f"[case] dequant {kind} {shape}", flush=True)
    w = (np.random.default_rng(N + K).standard_normal((N, K)) * 0.05).astype(np.float32)
    if kind in ("q8_0", "q4_0"):
        qt = oq.TYPE_Q8_0 if kind == "q8_0" else oq.TYPE_Q4_0
        blocks = oq.quantize_q8_0(w) if kind == "q8_0" else oq.quantize_q4_0(w)
        values = oq.dequantize(blocks, qt, K)
        rows, pad = torch.from_numpy(blocks), 6
        wrap = lambda t: kd_mm.QuantWeight(t, qt, K)
    else:
        rows = torch.from_numpy(w).to({"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}[kind])
        values, pad = rows.float().numpy(), 8
        wrap = lambda t: t
    expect = torch.from_numpy(oq.round_bf16(values)).to(torch.bfloat16)
    wide = torch.zeros((N, rows.shape[1] + pad), dtype=rows.dtype, device=DEV)
    wide[:, :rows.shape[1]] = rows.to(DEV)
    for src in (rows.to(DEV), wide[:, :rows.shape[1]]):
        weight = wrap(src)
        out = torch.full((N * K + 8,), 7.0, dtype=torch.bfloat16, device=DEV)
        view = kd_mm.w_view(weight)
        stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
        assert kd_mm._lib().kd_mm_dequant(ctypes.byref(view), ctypes.c_void_p(out.data_ptr()), N * K * 2, stream) == 0
        torch.cuda.synchronize()
        assert torch.equal(out[:N * K].cpu().view(torch.int16), expect.reshape(-1).view(torch.int16))
        assert bool((out[N * K:] == 7.0).all())
