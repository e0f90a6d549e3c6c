"""The C ABI's entry points captured in a HIP graph (torch.cuda.CUDAGraph):
each replay, with new inputs copied in eagerly between replays, gives the
bytes of the same calls made eagerly.  This covers the contract that the
entry points only enqueue work (no allocation, no host synchronisation, no
memset nodes): the general quantizer clears its block-max workspace with a
kernel on every replay, and the fused elementwise general path and the Gram
product's partial-tile flags likewise; the (1, 1) requantization epilogue,
the elementwise (1, 1) quantizer, the weight gradient's block maxima with
the requantization that starts from them, and the products of few tiles with
their device flags and partial sums are captured too."""
import numpy as np
import pytest
import torch

from oracle import qarr_oracle as O

pytestmark = pytest.mark.gpu


def _K():
    from pratchya_amd import _kernels
    return _kernels


def _same(a, b, what):
    """Bitwise equality of two tensors of one dtype and shape."""
    assert a.dtype == b.dtype and a.shape == b.shape, what
    assert torch.equal(a.contiguous().view(torch.uint8), b.contiguous().view(torch.uint8)), what


def test_graph_replays_match_eager():
    K = _K()
    gen = torch.Generator(device="cuda").manual_seed(41)
    M, Kd, N = 512, 1024, 768
    x = torch.empty((M, Kd), dtype=torch.bfloat16, device="cuda")
    w = torch.empty((Kd, N), dtype=torch.bfloat16, device="cuda")
    y = torch.empty((M, Kd), dtype=torch.bfloat16, device="cuda")

    def fill():
        x.copy_(torch.randn((M, Kd), generator=gen, device="cuda").to(torch.bfloat16))
        w.copy_((torch.randn((Kd, N), generator=gen, device="cuda") * 0.02).to(torch.bfloat16))
        y.copy_(torch.randn((M, Kd), generator=gen, device="cuda").to(torch.bfloat16))

    def work():
        xq = K.quantize(x, (1, 128))                                    # one-pass kernel
        wq = K.quantize(w, (128, 128))                                  # a workgroup per block, maxima in the workspace
        wf = K.quantize(w, (8, 32))                                     # general path: workspace cleared by a kernel
        wd = K.quantize_dequantize(w, (8, 32), torch.float32)           # the same, dequantized
        yq = K.quantize(y, (1, 128))
        a = K.operand_rows(*xq, (1, 128))
        b = K.operand_transposed(*wq, (128, 128))
        c = K.gemm_nt(a, b, torch.bfloat16)                            # block-scaled FP8 GEMM
        s = K.elementwise("add", xq, (1, 128), yq, (1, 128), (1, 128))  # fused, one pass
        d = K.elementwise("mul", xq, (1, 128), yq, (1, 128), (4, 64))   # fused, general path
        t = K.quantize_t128(x)                                          # transposed requantize
        q = K.dequantize(*xq, torch.float32, (1, 128))
        gr = K.gemm_bf16_gram(x)                                        # stream-K, flags cleared by a kernel
        ns = K.gemm_bf16_nt_ns(x, x, gr)                                # Newton-Schulz epilogue
        b11 = K.operand_transposed(*K.quantize(w, (128, 1)), (128, 1))
        o11 = K.gemm_nt_q11(a, b11, torch.bfloat16)                     # (1, 1) requantization epilogue
        x11 = K.quantize(x, (1, 1))                                     # elementwise (1, 1) kernel
        c32, bm = K.gemm_nt_blockmax(a, b)                              # block maxima from the epilogue
        wg = K.quantize_dequantize_premax(c32, bm, (128, 128), torch.bfloat16)
        return [*xq, *wq, *wf, *wd, c, *s, *d, *t, q, gr, ns, *o11, *x11, c32, bm, *wg]

    fill()
    torch.cuda.synchronize()
    work()                                   # warm up outside the capture
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        outs = work()
    for rep in range(3):
        fill()                               # eager work between replays
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        want = work()
        torch.cuda.synchronize()
        assert len(want) == len(outs)
        for i, (got, ref) in enumerate(zip(outs, want)):
            _same(got, ref, f"replay {rep}, output {i}")
    # and the replayed quantize is the oracle's
    xo = O.quantize_impl(x.float().cpu().numpy(), (1, 128))
    assert np.array_equal(outs[0].view(torch.uint8).cpu().numpy(), xo[0])


def test_graph_of_few_tile_products():
    """Split-K products, products of planes whose flags the device sets anew on
    every replay (a third piece that is zero or not, a cotangent that is finite
    or not), fine-block products and batched slices."""
    from pratchya_amd import optim
    from pratchya_amd import qarr as Q
    K = _K()
    gen = torch.Generator(device="cuda").manual_seed(43)
    M, Kd, N = 200, 1024, 512
    x = torch.empty((M, Kd), device="cuda")
    w = torch.empty((Kd, N), dtype=torch.bfloat16, device="cuda")
    g = torch.empty((M, N), dtype=torch.bfloat16, device="cuda")
    s = torch.empty((3, 128, 320), dtype=torch.bfloat16, device="cuda")

    def fill(rep):
        v = torch.randn((M, Kd), generator=gen, device="cuda")
        x.copy_(v.to(torch.bfloat16) if rep % 2 else v)
        w.copy_(torch.randn((Kd, N), generator=gen, device="cuda") * 0.02)
        g.copy_(torch.randn((M, N), generator=gen, device="cuda"))
        if rep == 2:
            g[3, 5], w[7, 9] = float("inf"), float("nan")
        s.copy_(torch.randn(s.shape, generator=gen, device="cuda"))

    def work():
        xq, wq = K.quantize(x, (1, 128)), K.quantize(w, (128, 128))
        a, b = K.operand_rows(*xq, (1, 128)), K.operand_transposed(*wq, (128, 128))
        c, f = K.gemm_t128(a, b), K.gemm_t128_fq(a, b, torch.bfloat16)
        grids = ((1, 128), (128, 128))
        gb = Q._plane_backward(g, (f[1], f[2], (1, 128)), xq + wq, grids, True, True)
        gf = Q._plane_backward(g.float(), (f[1], f[2], (1, 128)), xq + wq, grids, True, True)
        fine = Q._fine_forward(*K.quantize(x, (1, 16)), *K.quantize(w, (16, 16)), (1, 16), (16, 16))
        fq = K.quantize_dequantize(c, (1, 16), torch.bfloat16)
        ns = optim._newton_schulz_bf16(K.ns_normalize_batch(s), 2)
        return [c, *f, *gb, *gf, fine, *fq, K.matmul_f32(x, w), K.matmul_f32(x, w.float()), ns]

    fill(0)
    torch.cuda.synchronize()
    work()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        outs = work()
    for rep in range(4):
        fill(rep)
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        want = work()
        torch.cuda.synchronize()
        for i, (got, ref) in enumerate(zip(outs, want)):
            _same(got, ref, f"replay {rep}, output {i}")
