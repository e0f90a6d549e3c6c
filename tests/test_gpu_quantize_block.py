"""Quantization with a workgroup per block (grids whose block is 4096 to 32768
elements in rows of 64 or more) or per group (blocks of 16 x 16 and 32 x 32)
against the oracle and, bit for bit, against the flat kernels, which take the
outputs that start at no multiple of 16 bytes (and larger blocks anyway)."""
import numpy as np
import pytest
import torch

from oracle import qarr_oracle as O
from tests.helpers import assert_bytes_equal, assert_f32_bits_equal, assert_payload_equal, f32, u8

pytestmark = pytest.mark.gpu

# (shape, grid): rows not a multiple of a step, one row step, several slices,
# the widest and smallest blocks, one group over the array, one block per group
CASES = [((3, 256, 384), (128, 128)), ((200, 192), (100, 64)), ((64, 64), (64, 64)), ((130, 1024), (65, 128)),
         ((256, 512), (128, 512)), ((48, 1024), (16, 256)), ((1024, 64), (1024, 64)), ((1024, 1024), (128, 128)),
         ((96, 128), (32, 128)), ((255, 256), (255, 256)),
         # groups of 16 blocks of 16 x 16: in one row of blocks, across two, several rows, several slices
         ((16, 256), (16, 16)), ((32, 384), (16, 16)), ((256, 48), (16, 16)), ((256, 16), (16, 16)),
         ((3, 64, 320), (16, 16)), ((208, 256), (16, 16)), ((16, 240), (16, 16)),
         # groups of 64 blocks of 32 x 32, and fewer blocks in a group
         ((32, 2048), (32, 32)), ((256, 256), (32, 32)), ((2, 64, 3072), (32, 32)), ((2048, 32), (32, 32)),
         ((320, 640), (32, 32))]


def _values(shape, dtype, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    x = torch.randn(shape, generator=g, device="cuda") * torch.exp2(
        torch.randint(-12, 13, shape[:-1] + (1,), generator=g, device="cuda").float())
    x = x.view(-1, shape[-1])
    x[:, 5] = 0.0
    if x.shape[0] >= 200:
        x[: x.shape[0] // 2, : shape[-1] // 2] *= 1e-12
        x[-1, -1], x[-2, 0] = float("inf"), float("nan")
    return x.view(shape).to(dtype)


def _unaligned(shape, dtype):
    """A buffer that the kernels of 16-byte stores do not take."""
    n = 1
    for d in shape:
        n *= d
    return torch.empty(n + 1, dtype=dtype, device="cuda")[1:].view(shape)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("shape,grid", CASES, ids=lambda v: "x".join(map(str, v)))
def test_block_per_workgroup(shape, grid, dtype):
    from pratchya_amd import _kernels as K
    x = _values(shape, dtype, 7)
    q, s8, s32 = K.quantize(x, grid)
    flat = (_unaligned(shape, torch.uint8), torch.empty_like(s8), torch.empty_like(s32))
    assert flat[0].data_ptr() % 16
    for got, want in zip(K.quantize(x, grid, out=flat), (q, s8, s32)):
        assert_bytes_equal(u8(got.contiguous().view(torch.uint8)), u8(want.contiguous().view(torch.uint8)), "flat")
    wq, we, wg = O.quantize_impl(f32(x), grid)
    assert_bytes_equal(u8(s8).reshape(-1), we.view(np.uint8).reshape(-1), "e8m0")
    assert_f32_bits_equal(f32(s32).reshape(-1), wg.reshape(-1), "group maxima")
    assert_payload_equal(u8(q), wq.view(np.uint8), "payload")
    for out in (torch.bfloat16, torch.float32):
        for fix in (False, True):
            a = K.quantize_dequantize(x, grid, out, fix)
            flat = (_unaligned(shape, out), torch.empty_like(a[1]), torch.empty_like(a[2]))
            assert flat[0].data_ptr() % 16
            for got, want in zip(a, K.quantize_dequantize(x, grid, out, fix, out=flat)):
                assert torch.equal(got.contiguous().view(torch.uint8), want.contiguous().view(torch.uint8))
            e = np.where(we.view(np.uint8) == 0xFF, np.uint8(0x7F), we.view(np.uint8)) if fix else we
            want = O.dequantize_impl(wq, e, wg, "float32" if out == torch.float32 else "bfloat16", grid)
            want = want if out == torch.float32 else O.bf16_bits_to_f32(want)
            assert_f32_bits_equal(f32(a[0]), want, "fake quantization")


@pytest.mark.parametrize("ids_shape,out_grid", [((256,), (128, 128)), ((2, 192), (64, 64)), ((100,), (50, 128)),
                                                ((640,), (128, 256))])
def test_gathered_rows(ids_shape, out_grid):
    """Looked-up rows requantized with a workgroup per block against the rows'
    values quantized by themselves; indices out of range, negative and equal."""
    from pratchya_amd import _kernels as K
    table = K.quantize(_values((384, 512), torch.bfloat16, 3), (128, 128))
    ids = torch.randint(-384, 384, ids_shape, device="cuda", generator=torch.Generator(device="cuda").manual_seed(1))
    ids.view(-1)[:4] = torch.tensor([0, 383, 100000, -100000], device="cuda")
    rows = K.gather_dequantize(*table, (128, 128), ids, torch.float32)
    for got, want in zip(K.gather_quantize(*table, (128, 128), ids, out_grid), K.quantize(rows, out_grid)):
        assert torch.equal(got.contiguous().view(torch.uint8), want.contiguous().view(torch.uint8))


# (both sides of the lines between the kernels: groups of 32 x 32 blocks for f32
# results, a block's bytes, blocks for each CU, elements in all)
LINES = [((2048, 4096), (32, 32)), ((2048, 4064), (32, 32)), ((768, 512), (192, 128)), ((800, 512), (200, 128)),
         ((4096, 1024), (256, 64)), ((3840, 1088), (256, 64)), ((4096, 4096), (64, 64)), ((4096, 4160), (64, 64)),
         ((4096, 4096), (64, 256)), ((8192, 4096), (64, 512)), ((8192, 8192), (128, 128)), ((8192, 8320), (128, 128))]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("shape,grid", LINES, ids=lambda v: "x".join(map(str, v)))
def test_lines_of_the_dispatch(shape, grid, dtype):
    from pratchya_amd import _kernels as K
    x = _values(shape, dtype, 8)
    got = K.quantize(x, grid)
    flat = (_unaligned(shape, torch.uint8), torch.empty_like(got[1]), torch.empty_like(got[2]))
    K.quantize(x, grid, out=flat)
    assert all(torch.equal(a.view(torch.uint8), b.view(torch.uint8)) for a, b in zip(got, flat))
    for out in (torch.bfloat16, torch.float32):
        got = K.quantize_dequantize(x, grid, out, True)
        flat = (_unaligned(shape, out), torch.empty_like(got[1]), torch.empty_like(got[2]))
        K.quantize_dequantize(x, grid, out, True, out=flat)
        assert all(torch.equal(a.view(torch.uint8), b.view(torch.uint8)) for a, b in zip(got, flat))
