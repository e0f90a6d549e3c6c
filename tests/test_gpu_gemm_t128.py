"""The 128-row-tile GEMM and the planes of its bf16 operands, at the edges of
its tiles (128 / 32 rows, 128 columns), its K slices and its scale spans, against
float64 products of the dequantized operands.

Tolerances: products of bf16 values are exact in f32, so a sum of K of them is
within K * 2^-24 of the sum of their magnitudes in any order; over random signs
the relative Frobenius error stays well below 2e-6 at these K (the f32 GEMM
tests' bound is 1e-5).
"""
import pytest
import torch

pytestmark = pytest.mark.gpu
TOL = 2e-6


def _K():
    from pratchya_amd import _kernels
    return _kernels


def _randn(shape, seed, dtype=torch.float32, scale=1.0):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return (torch.randn(shape, generator=g, device="cuda") * scale).to(dtype)


def _rel(a, b):
    return float((a.double() - b).norm() / b.norm())


@pytest.mark.parametrize("M,N,Kd", [(1, 8, 64), (32, 128, 128), (33, 136, 64), (127, 260, 192), (129, 128, 4096),
                                    (1000, 2944, 2176), (640, 384, 12288)])
def test_bf16_product(M, N, Kd):
    K = _K()
    a, b = _randn((1, M, Kd), 1, torch.bfloat16), _randn((1, N, Kd), 2, torch.bfloat16)
    ref = a[0].double() @ b[0].double().T
    c = K.gemm_planes(a, b, [(0, 0)], False)
    assert _rel(c, ref) <= TOL
    if M % 8 == 0 and M > 32 and N % 8 == 0:      # K-major operands: the same sums
        assert torch.equal(c, K.gemm_planes(a.transpose(1, 2).contiguous(), b.transpose(1, 2).contiguous(), [(0, 0)],
                                            True))


@pytest.mark.parametrize("rows,Kd,N,blk,dtype", [
    (100, 256, 512, 16, torch.bfloat16), (300, 1024, 768, 128, torch.bfloat16), (64, 2176, 2944, 128, torch.bfloat16),
    (257, 512, 640, 32, torch.bfloat16), (130, 512, 1024, 128, torch.float32), (65, 1280, 640, 16, torch.float32)])
def test_backward_products(rows, Kd, N, blk, dtype):
    """Both f32 cotangents of a quantized product whose output scales the
    cotangent carries, against float64 (blocks of very different sizes, group
    maxima that change along the contraction); bf16 sources need two pieces of
    x, f32 ones three."""
    from pratchya_amd import qarr as Q
    K = _K()
    w = (_randn((Kd, N), 3) * torch.exp(_randn((Kd, N), 4)) * 0.02).to(dtype)
    xq = K.quantize(_randn((rows, Kd), 5, dtype), (1, blk))
    wq = K.quantize(w, (blk, blk))
    oq = K.quantize(_randn((rows, N), 6, scale=3.0), (1, blk))
    g = _randn((rows, N), 7, dtype)
    g1 = K.dequantize_bwd(g, oq[1], oq[2], (1, blk)).double()
    wd, xd = K.dequantize(*wq, torch.float32, (blk, blk)).double(), K.dequantize(*xq, torch.float32, (1, blk)).double()
    gx, gw = Q._plane_backward(g, (oq[1], oq[2], (1, blk)), xq + wq, ((1, blk), (blk, blk)), True, True)
    assert _rel(gx, g1 @ wd.T) <= TOL and _rel(gw, xd.T @ g1) <= TOL


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_backward_products_non_finite(dtype):
    """inf and NaN cotangents, a zero weight group and an x too large to
    dequantize: the same elements are inf, -inf and NaN as in the f32 products
    of the dequantized operands."""
    from pratchya_amd import qarr as Q
    K = _K()
    rows, Kd, N, blk = 192, 256, 384, 128
    x, w, g = _randn((rows, Kd), 1, dtype), _randn((Kd, N), 2, dtype), _randn((rows, N), 3, dtype)
    x[5, 3], w[:128] = 3e38, 0.0
    g[7, 9], g[70, 11], g[100, 300] = float("inf"), float("-inf"), float("nan")
    xq, wq = K.quantize(x, (1, blk)), K.quantize(w, (blk, blk))
    gx, gw = Q._plane_backward(g, None, xq + wq, ((1, blk), (blk, blk)), True, True)
    xd, wd = K.dequantize(*xq, torch.float32, (1, blk)), K.dequantize(*wq, torch.float32, (blk, blk))
    for got, ref in ((gx, K.matmul_f32(g, wd, False, True)), (gw, K.matmul_f32(xd, g, True, False))):
        assert torch.equal(torch.nan_to_num(got, 0.0, 1.0, -1.0)[~torch.isfinite(ref)],
                           torch.nan_to_num(ref, 0.0, 1.0, -1.0)[~torch.isfinite(ref)])
        assert torch.equal(torch.isfinite(got), torch.isfinite(ref))


def test_planes_sum_to_the_value():
    K = _K()
    x = _randn((130, 512), 1) * torch.exp(4 * _randn((130, 512), 2))
    q = K.quantize(x, (1, 32))
    d = K.dequantize(*q, torch.float32, (1, 32))
    flags = torch.zeros(2, dtype=torch.int32, device="cuda")
    p = K.planes(K.PLANE_SPLIT3, *q, (1, 32), flags, pad=64)
    assert p.shape == (3, 192, 512) and not p[:, 130:].any() and flags.tolist() == [1, 0]
    assert torch.equal(p[:, :130].double().sum(0), d.double())
    assert torch.equal(K.planes(K.PLANE_SPLIT4, d, None, None, None)[:3].double().sum(0), d.double())
    # the power-of-two plane times the group maximum's mantissa is the value
    pw = K.planes(K.PLANE_POW2, *q, (1, 32))[0].double()
    mant = torch.frexp(q[2].flatten().double())[0] * 2
    assert torch.allclose(pw * mant.repeat_interleave(64).view(130, 512), d.double(), rtol=2 ** -23, atol=0)
    flags.zero_()
    K.planes(K.PLANE_SPLIT3, *K.quantize(x.to(torch.bfloat16), (1, 32)), (1, 32), flags)
    assert flags.tolist() == [0, 0]              # bf16 group maxima: no third piece


@pytest.mark.parametrize("M,N,Kd,grid", [
    (1, 256, 128, (128, 128)), (32, 1024, 4096, (128, 128)), (33, 384, 640, (128, 128)), (7, 512, 2176, (128, 1)),
    (129, 272, 2176, (128, 8)), (300, 2944, 512, (128, 1)), (512, 1024, 1152, (128, 64))])
def test_fp8_product(M, N, Kd, grid):
    """gemm_t128 on (1, 128) activations and weight grids whose group maxima
    change along K, against the 256x256 kernel (the same MFMAs, summed in
    another order: f32 rounding, bound as above) and float64 (the f32 tolerance
    of the FP8 GEMM tests)."""
    K = _K()
    x = _randn((M, Kd), 1) * torch.exp(2 * _randn((M, 1), 2))
    w = _randn((Kd, N), 3, scale=0.02) * torch.exp(_randn((Kd, N), 4))
    xq, wq = K.quantize(x, (1, 128)), K.quantize(w, grid)
    a, b = K.operand_rows(*xq, (1, 128)), K.operand_transposed(*wq, grid)
    ref = K.dequantize(*xq, torch.float32, (1, 128)).double() @ K.dequantize(*wq, torch.float32, grid).double()
    c = K.gemm_t128(a, b, torch.float32)
    assert _rel(c, ref) <= 1e-3 and _rel(c, K.gemm_nt(a, b, torch.float32).double()) <= TOL
    assert _rel(K.gemm_t128(a, b, torch.bfloat16), c.double()) <= 2.0 ** -8
    if grid[1] % 128 == 0:                        # as the weight's rows (dgrad): group maxima per 128 rows
        g = K.quantize(_randn((M, N), 5), (1, 128))
        op_w = K.operand_rows(*wq, grid)
        og = K.operand_rows(*g, (1, 128))
        if N % 128 == 0:
            assert _rel(K.gemm_t128(og, op_w, torch.float32), K.gemm_nt(og, op_w, torch.float32).double()) <= TOL


@pytest.mark.parametrize("rows", [1, 32, 33, 200])
@pytest.mark.parametrize("grid,N", [((128, 128), 1024), ((128, 1), 528)])
def test_linear_of_few_rows(rows, grid, N):
    """A Linear of few rows (fused requantization asked for, the product on
    gemm_t128): the same output as its steps."""
    from pratchya_amd import qarr as Q
    K = _K()
    x, w = _randn((rows, 2048), 1, torch.bfloat16), _randn((2048, N), 2, torch.bfloat16, 0.02)
    W = Q.QArrayImpl(w, grid)
    y = (Q.QArrayImpl(x, (1, 128)) @ W).astype(torch.bfloat16)
    xq = K.quantize(x, (1, 128))
    c = K.gemm_t128(K.operand_rows(*xq, (1, 128)), K.operand_transposed(*W._tree_flatten()[0], grid), torch.float32)
    assert torch.equal(y, K.quantize_dequantize(c, (1, grid[1]), torch.bfloat16)[0])


@pytest.mark.parametrize("shape", [(64, 64), (256, 512), (320, 1024), (1024, 192), (2048, 2304), (2304, 2048)])
def test_newton_schulz_of_few_tiles(shape):
    """Sides at the dispatch's edges against the same iteration in float64 (the
    bf16 tolerance of the optimizer tests)."""
    from pratchya_amd.optim import newton_schulz
    g = _randn(shape, 1, torch.bfloat16)
    x = g.double() / g.double().norm()
    x = x.T if shape[0] > shape[1] else x
    for _ in range(5):
        x = 1.5 * x - 0.5 * (x @ x.T) @ x
    assert _rel(newton_schulz(g), x.T if shape[0] > shape[1] else x) <= 3e-2
    K = _K()
    a = K.gemm_planes(g[None], g[None], [(0, 0)], False, torch.bfloat16)
    assert torch.equal(a, a.T)


@pytest.mark.parametrize("rows,Kd,N,blk,dtype", [
    (1, 64, 16, 16, torch.bfloat16), (32, 128, 640, 16, torch.bfloat16), (33, 192, 96, 32, torch.bfloat16),
    (129, 576, 2944, 16, torch.float32), (300, 1088, 352, 32, torch.float32), (520, 4096, 128, 16, torch.bfloat16)])
def test_fine_block_product(rows, Kd, N, blk, dtype):
    """The forward product of blocks of 16 and 32 against float64, group maxima
    of very different sizes, groups of the weight that straddle its block rows
    (2944 / 16 = 184 blocks), 3-D activations, and rows of zeros, inf and NaN."""
    from pratchya_amd import qarr as Q
    K = _K()
    x = (_randn((rows, Kd), 1) * torch.exp(3 * _randn((rows, Kd // blk), 2)).repeat_interleave(blk, 1)).to(dtype)
    w = (_randn((Kd, N), 3) * torch.exp(_randn((Kd, N), 4)) * 0.02).to(dtype)
    xq, wq = K.quantize(x, (1, blk)), K.quantize(w, (blk, blk))
    xd, wd = K.dequantize(*xq, torch.float32, (1, blk)), K.dequantize(*wq, torch.float32, (blk, blk))
    c = Q._fine_forward(*xq, *wq, (1, blk), (blk, blk))
    assert _rel(c, xd.double() @ wd.double()) <= TOL
    if rows % 3 == 0:
        x3 = K.quantize(x.view(3, rows // 3, Kd), (1, blk))
        assert torch.equal(Q._matmul_forward(*x3, *wq, (1, blk), (blk, blk)).view(rows, N), c)
    if rows > 4:
        x[0], x[1, 3], x[2, 5], x[3, 7] = 0.0, float("inf"), float("nan"), 3e38
        xq = K.quantize(x, (1, blk))
        c = Q._fine_forward(*xq, *wq, (1, blk), (blk, blk))
        ref = K.matmul_f32(K.dequantize(*xq, torch.float32, (1, blk)), wd)
        assert torch.equal(torch.isfinite(c), torch.isfinite(ref)) and not c[0].any()


@pytest.mark.parametrize("xdt", ["bf16", "f32"])
@pytest.mark.parametrize("tgrid", [(1, 8), (1, 16), (1, 32), (1, 64)])
@pytest.mark.parametrize("out", ["bfloat16", "float32"])
@pytest.mark.parametrize("fix_nan", [False, True])
def test_fake_quantization_of_narrow_row_blocks(xdt, tgrid, out, fix_nan):
    """The one-pass fake quantization of (1, b) grids, bit for bit against the
    oracle on the edge values (zeros, clamped groups, overflow, NaN, inf,
    subnormals, quotients next to bf16 midpoints) and on a partial last wave."""
    import numpy as np

    from oracle import qarr_oracle as O
    from tests.helpers import to_dev_bf16, to_dev_f32
    from tests.test_gpu_qdq import check, edge_tensor
    x = edge_tensor(xdt)
    dev = to_dev_bf16(O.f32_to_bf16_bits(x)) if xdt == "bf16" else to_dev_f32(x)
    check(dev, x, tgrid, out, fix_nan, f"edge {xdt} {tgrid}->{out} fix {fix_nan}")
    y = np.random.default_rng(3).standard_normal((5, 192)).astype(np.float32)
    y = O.bf16_round(y) if xdt == "bf16" else y
    dev = to_dev_bf16(O.f32_to_bf16_bits(y)) if xdt == "bf16" else to_dev_f32(y)
    check(dev, y, tgrid, out, fix_nan, f"ragged {xdt} {tgrid}->{out} fix {fix_nan}")


@pytest.mark.parametrize("a_t", [False, True])
@pytest.mark.parametrize("b_t", [False, True])
@pytest.mark.parametrize("M,N,Kd", [(40, 8, 64), (264, 136, 192), (136, 520, 200), (1024, 1024, 1024)])
@pytest.mark.parametrize("bdt", [torch.float32, torch.bfloat16])
def test_matmul_f32_layouts(a_t, b_t, M, N, Kd, bdt):
    """f32 products of few tiles from planes in the operands' own layouts (and
    the packed pieces where a layout does not fit: K = 200), with an inf in each
    operand: finite elements to f32 accuracy, the others where float64 has them."""
    K = _K()
    a = _randn((Kd, M) if a_t else (M, Kd), 1) * torch.exp(_randn((1,), 2))
    b = _randn((N, Kd) if b_t else (Kd, N), 3, bdt)
    if Kd == 192:
        a[3, 5], b[7, 2] = float("inf"), float("-inf")
    ref = (a.T if a_t else a).double() @ (b.T if b_t else b).double()
    c = K.matmul_f32(a, b, a_t, b_t)
    ok = torch.isfinite(ref)
    assert torch.equal(torch.isfinite(c), ok) and _rel(torch.where(ok, c, 0.0), torch.where(ok, ref, 0.0)) <= TOL
    if a_t and not b_t and bdt == torch.float32:
        assert _rel(K.matmul_f32(a, a, True, False), a.double().T @ a.double()) <= TOL or Kd == 192


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("shape", [(4300, 256, 2048), (4353, 384, 1040), (70000, 128, 48)])
def test_one_by_one_epilogue_without_scales(shape, dt):
    """The (1, 1) epilogue with its scale arrays left out stores the same values."""
    K = _K()
    M, Kd, N = shape
    a = K.operand_rows(*K.quantize(_randn((M, Kd), 1, torch.bfloat16), (1, 128)), (1, 128))
    b = K.operand_transposed(*K.quantize(_randn((Kd, N), 2, torch.bfloat16) * 0.02, (128, 1)), (128, 1))
    y, s8, s32 = K.gemm_nt_q11(a, b, dt)
    z, n8, n32 = K.gemm_nt_q11(a, b, dt, scales=False)
    assert n8 is None and n32 is None and s8 is not None and s32 is not None
    assert torch.equal(y, z)


def test_batched_slices():
    """Batches of products and normalizations against their slices, K split or
    not, and a stacked optimizer leaf in runs of one layer against all at once."""
    from pratchya_amd import optim
    K = _K()
    for shape in [(3, 320, 512), (2, 1024, 4096), (5, 256, 64)]:
        x = _randn(shape, 1, torch.bfloat16)
        for km in (False, True):
            c = K.gemm_planes_batch(x, x, km, torch.bfloat16)
            assert torch.equal(c, c.transpose(1, 2))
            ref = (x.transpose(1, 2).float() @ x.float()) if km else (x.float() @ x.transpose(1, 2).float())
            assert _rel(c.float(), ref.double()) <= 2.0 ** -8
        a = K.gemm_planes_batch(x, x, False, torch.bfloat16)
        y = K.gemm_planes_batch(a, x, False, torch.bfloat16, x=x, b_k_major=True)
        for i in range(shape[0]):
            p = (a[i].float() @ x[i].float()).to(torch.bfloat16)
            assert _rel(y[i].float(), K.ns_combine(x[i], p).double()) <= 2.0 ** -6
            assert torch.equal(K.ns_normalize_batch(x)[i], K.ns_normalize(x[i]))
    grid, sh = (64, 64), (3, 128, 192)
    mom, par = (K.quantize(_randn(sh, s) * 1e-3, grid) for s in (4, 5))
    args = (("layers",), _randn(sh, 6, torch.bfloat16), mom, par, grid, 0.9, 0.99, 5, 3e-4, 0.02, 0.1)
    one, prev = optim._quantized_stack_step(*args), optim._STACK_ELEMENTS
    try:
        optim._STACK_ELEMENTS = 1
        runs = optim._quantized_stack_step(*args)
    finally:
        optim._STACK_ELEMENTS = prev
    assert _rel(runs[0].float(), one[0].double()) <= 3e-2
    for p, q in zip(one[1], runs[1]):
        assert p.dtype == q.dtype and torch.equal(p.view(torch.uint8), q.view(torch.uint8))


@pytest.mark.parametrize("lead,Kd,N", [((1,), 128, 1024), ((4,), 4096, 4096), ((8,), 128, 128), ((33,), 256, 1024),
                                       ((1000,), 2176, 2944), ((2, 8), 512, 384), ((640,), 4096, 1152)])
@pytest.mark.parametrize("dt,fix_nan", [(torch.bfloat16, False), (torch.float32, True)])
def test_requantized_sum_of_slices(lead, Kd, N, dt, fix_nan):
    """The requantization that sums the K slices itself: the bits of the
    reduced product's, scales stored or not."""
    K = _K()
    rows = 1
    for d in lead:
        rows *= d
    x = _randn((rows, Kd), 30, torch.bfloat16, 3.0)
    x[0, :128] = 0                                   # a block of zeros
    if rows > 4:
        x[3] = 0
        x[4, 5] = float("nan") if fix_nan else float("inf")
    a = K.operand_rows(*K.quantize(x, (1, 128)), (1, 128))
    b = K.operand_transposed(*K.quantize(_randn((Kd, N), 31, torch.bfloat16, 0.02), (128, 128)), (128, 128))
    ref = K.quantize_dequantize(K.gemm_t128(a, b, torch.float32).view(lead + (N,)), (1, 128), dt, fix_nan)
    got = K.gemm_t128_fq(a, b, dt, fix_nan, lead)
    bare = K.gemm_t128_fq(a, b, dt, fix_nan, lead, scales=False)
    assert got[0].shape == (rows, N) and [t.shape for t in got[1:]] == [t.shape for t in ref[1:]]
    for r, t in zip(ref, got):
        assert torch.equal(r.reshape(-1).view(torch.uint8), t.reshape(-1).view(torch.uint8))
    assert torch.equal(bare[0].view(torch.uint8), got[0].view(torch.uint8)) and bare[1:] == (None, None)


def test_requantized_sum_refusals():
    K = _K()
    a = K.operand_rows(*K.quantize(_randn((5, 256), 1, torch.bfloat16), (1, 128)), (1, 128))
    b = K.operand_transposed(*K.quantize(_randn((256, 384), 2, torch.bfloat16), (128, 128)), (128, 128))
    with pytest.raises(K.PratchyaUnsupported):
        K.gemm_t128_fq(a, b, torch.bfloat16)         # 15 blocks: not whole groups of 8


def _shifted(t, n):
    """A copy of ``t`` that starts n elements into its buffer."""
    buf = torch.empty(t.numel() + n, dtype=t.dtype, device=t.device)
    return buf[n:].copy_(t.reshape(-1)).view(t.shape)


def test_scales_inside_larger_arrays():
    """Scale arrays that start at no multiple of 16 (of 4) bytes."""
    from pratchya_amd import qarr as Q
    K = _K()
    xq, wq = K.quantize(_randn((100, 512), 1), (1, 16)), K.quantize(_randn((512, 256), 2), (16, 16))
    c = Q._fine_forward(*xq, *wq, (1, 16), (16, 16))
    at = xq[0], _shifted(xq[1].view(torch.uint8), 1).view(xq[1].dtype), _shifted(xq[2], 1)
    assert at[2].data_ptr() % 16 and torch.equal(Q._fine_forward(*at, *wq, (1, 16), (16, 16)), c)
    xq, wq = K.quantize(_randn((100, 512), 3), (1, 128)), K.quantize(_randn((512, 256), 4), (128, 128))
    w = K.operand_transposed(*wq, (128, 128))
    c = K.gemm_t128(K.operand_rows(*xq, (1, 128)), w)
    at = xq[0], _shifted(xq[1].view(torch.uint8), 1).view(xq[1].dtype), _shifted(xq[2], 1)
    assert at[1].data_ptr() % 4 and torch.equal(K.gemm_t128(K.operand_rows(*at, (1, 128)), w), c)


@pytest.mark.parametrize("rows", [5, 33, 200])
def test_payload_at_any_offset(rows):
    """A payload of fewer than 256 rows that starts at no multiple of 16 bytes, as
    the kernels of more tiles take it (they copy it): the same products, on the
    split-K kernel and its requantizing form, and through the public product."""
    from pratchya_amd import qarr as Q
    K = _K()
    xq, wq = K.quantize(_randn((rows, 512), 3), (1, 128)), K.quantize(_randn((512, 1024), 4), (128, 128))
    at = (_shifted(xq[0].view(torch.uint8), 8).view(xq[0].dtype),) + xq[1:]
    assert at[0].data_ptr() % 16
    w = K.operand_transposed(*wq, (128, 128))
    a, b = K.operand_rows(*xq, (1, 128)), K.operand_rows(*at, (1, 128))
    assert torch.equal(K.gemm_t128(b, w), K.gemm_t128(a, w))
    for got, want in zip(K.gemm_t128_fq(b, w, torch.bfloat16), K.gemm_t128_fq(a, w, torch.bfloat16)):
        assert torch.equal(got.view(torch.uint8), want.view(torch.uint8))
    mk = Q.QArrayImpl._tree_unflatten
    W = mk((True, (128, 128)), wq)
    for dt in (torch.bfloat16, torch.float32):
        y, z = ((mk((True, (1, 128)), t) @ W).astype(dt) for t in (xq, at))
        assert torch.equal(y, z)


def test_cotangent_scaled_once(monkeypatch):
    """The default backward of an output head ((1, 1) output blocks, a weight in
    one-column blocks): the cotangent goes through dequantize_impl_bwd once,
    whichever products take it."""
    from pratchya_amd import qarr as Q
    K = _K()
    x, w = _randn((300, 256), 1, torch.bfloat16).requires_grad_(), _randn((256, 640), 2, torch.bfloat16, 0.02)
    w.requires_grad_()
    y = (Q.QArrayImpl(x, (1, 128)) @ Q.QArrayImpl(w, (128, 1))).astype(torch.bfloat16)
    calls, scale = [], K.dequantize_bwd
    monkeypatch.setattr(K, "dequantize_bwd", lambda *a: calls.append(a[0].shape) or scale(*a))
    torch.autograd.grad(y, (x, w), torch.ones_like(y))
    assert len(calls) == 1



@pytest.mark.parametrize("M,N,Kd,a_t,b_t", [(100, 520, 192, True, False), (96, 524, 192, False, False),
                                            (96, 102, 192, False, True), (96, 102, 192, False, False),
                                            (96, 520, 200, False, False)])
@pytest.mark.parametrize("bdt", [torch.float32, torch.bfloat16])
def test_no_planes_for_refused_products(M, N, Kd, a_t, b_t, bdt, monkeypatch):
    """An f32 product whose planes the 128x128 kernel would refuse (a side of its
    K-major operands no multiple of 8, an N no multiple of 4) writes none."""
    K = _K()
    a, b = _randn((Kd, M) if a_t else (M, Kd), 1), _randn((N, Kd) if b_t else (Kd, N), 2, bdt)
    calls, planes = [], K.planes
    monkeypatch.setattr(K, "planes", lambda *a, **k: calls.append(a[0]) or planes(*a, **k))
    c = K.matmul_f32(a, b, a_t, b_t)
    ref = (a.T if a_t else a).double() @ (b.T if b_t else b).double()
    assert not calls and _rel(c, ref) <= TOL


@pytest.mark.parametrize("M,N,Kd,adt,bdt,planes,few", [
    (256, 256, 256, "f", "b", 0, False), (1024, 1024, 128, "f", "b", 0, True), (256, 256, 384, "f", "b", 2, True),
    (256, 256, 64, "f", "f", 2, True), (2048, 2048, 448, "b", "b", 0, True), (2048, 2048, 512, "b", "b", 0, False),
    (2048, 2048, 960, "b", "b", 0, False), (2048, 2048, 1024, "b", "b", 0, True), (4096, 2048, 448, "b", "b", 0, False),
    (4096, 2048, 512, "b", "b", 0, True), (512, 1024, 256, "b", "f", 0, False), (40, 8192, 768, "b", "b", 0, True),
    (264, 136, 600, "b", "b", 0, True)])
def test_routes_of_short_products(M, N, Kd, adt, bdt, planes, few, monkeypatch):
    """On both sides of the lines that choose an f32 product's tiles: the route,
    and the product against float64."""
    K = _K()
    dt = {"f": torch.float32, "b": torch.bfloat16}
    a, b = _randn((M, Kd), 1, dt[adt]), _randn((Kd, N), 2, dt[bdt])
    calls = {"planes": 0, "gemm_planes": 0, "gemm_bf16_nt": 0}
    for name in calls:
        def spy(*args, _f=getattr(K, name), _n=name, **kw):
            calls[_n] += 1
            return _f(*args, **kw)
        monkeypatch.setattr(K, name, spy)
    c = K.matmul_f32(a, b)
    assert calls == {"planes": planes, "gemm_planes": int(few), "gemm_bf16_nt": int(not few)}
    assert _rel(c, a.double() @ b.double()) <= TOL


@pytest.mark.parametrize("M,Kd,sr", [(100, 768, 8), (7, 768, 8), (100, 640, 0), (33, 1152, 12), (100, 1024, 8)])
def test_strided_scale_rows(M, Kd, sr):
    """The C entry on rows of e8m0 bytes in wider rows (or one row's shared by
    all: sr 0) whose last row ends with its last used byte: the product of the
    same scales packed, all K steps of the last rows included."""
    K = _K()
    lib = K._lib.load()
    N, nk, kg = 256, Kd // 128, 2
    gen = torch.Generator(device="cuda").manual_seed(9)
    a = K.quantize(_randn((M, Kd), 1), (1, 128))[0]
    rows = M if sr else 1
    e8 = torch.randint(121, 128, (rows, nk), generator=gen, device="cuda", dtype=torch.uint8)
    g32 = torch.rand((rows, -(-nk // kg)), generator=gen, device="cuda") + 0.5
    w = K.operand_transposed(*K.quantize(_randn((Kd, N), 2), (128, 128)), (128, 128))

    def product(e, g, a_sr, a_kg):
        c = torch.empty((M, N), device="cuda")
        ws_bytes = lib.pratchya_gemm_t128_workspace_bytes(M, N, nk, 1)
        ws = torch.empty(max(ws_bytes, 1), dtype=torch.uint8, device="cuda")
        K._lib.check(lib.pratchya_gemm_bs_t128(
            K._ptr(a), Kd, K._ptr(e), K._ptr(g), 1, a_sr, 1, a_kg, K._ptr(w.payload), Kd, K._ptr(w.sc8), K._ptr(w.sc32),
            *w.desc, M, N, Kd, K._ptr(c), N, K._dtype_code(c.dtype), K._ptr(ws), ws_bytes, K._stream(a)), "gemm_t128")
        return c

    wide = torch.full(((rows - 1) * sr + nk,), 255, dtype=torch.uint8, device="cuda")
    gw = torch.full((wide.numel() // kg + 1,), float("nan"), device="cuda")
    for r in range(rows):
        wide[r * sr:r * sr + nk] = e8[r]
        gw[r * sr // kg:r * sr // kg + g32.shape[1]] = g32[r]
    # packed, one block per group
    ep = e8.expand(M, nk).contiguous()
    gp = g32.repeat_interleave(kg, 1)[:, :nk].expand(M, nk).contiguous()
    assert _rel(product(wide, gw, sr, kg), product(ep, gp, nk, 1).double()) <= TOL


def test_input_gradient_of_a_non_finite_weight():
    """A weight too large to dequantize (inf): an f32 cotangent's products with it
    are inf, -inf and NaN where the f32 products of the dequantized operands are
    (a zero piece of a finite value meets no inf)."""
    from pratchya_amd import qarr as Q
    K = _K()
    rows, Kd, N, blk = 192, 256, 384, 128
    x, w, g = _randn((rows, Kd), 1), _randn((Kd, N), 2), _randn((rows, N), 3)
    g = torch.where(torch.rand((rows, N), device="cuda", generator=torch.Generator(device="cuda").manual_seed(4)) < 0.3,
                    g.to(torch.bfloat16).float(), g)        # values of one piece among those of three
    w[3, 5], w[200, 300] = 3e38, -3e38
    xq, wq = K.quantize(x, (1, blk)), K.quantize(w, (blk, blk))
    wd = K.dequantize(*wq, torch.float32, (blk, blk))
    assert int(torch.isinf(wd).sum()) == 2
    gx = Q._plane_backward(g, None, xq + wq, ((1, blk), (blk, blk)), True, False)[0]
    ref = g.double() @ wd.double().T
    assert torch.equal(torch.isnan(gx), torch.isnan(ref)) and torch.equal(torch.isposinf(gx), torch.isposinf(ref))
    fin = torch.isfinite(ref)
    assert torch.equal(torch.isfinite(gx), fin) and not bool(fin.all())
    assert _rel(torch.where(fin, gx, 0.0), torch.where(fin, ref, 0.0)) <= TOL


@pytest.mark.parametrize("rows", [1, 32, 33, 200])
@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
def test_few_row_head_without_scales(rows, dt):
    """The output head's product of few rows without its scale arrays: the same
    values, and no scale arrays."""
    K = _K()
    a = K.operand_rows(*K.quantize(_randn((rows, 2048), 1, torch.bfloat16), (1, 128)), (1, 128))
    b = K.operand_transposed(*K.quantize(_randn((2048, 528), 2, torch.bfloat16, 0.02), (128, 1)), (128, 1))
    y, s8, s32 = K.gemm_nt_q11(a, b, dt, few=True)
    z, n8, n32 = K.gemm_nt_q11(a, b, dt, few=True, scales=False)
    assert s8 is not None and s32 is not None and n8 is None and n32 is None and torch.equal(y, z)
