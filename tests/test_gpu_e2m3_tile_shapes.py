"""The FP6 GEMM at sizes that reach each of its tile shapes (the comments name them: K-split or 2 x 2 waves, row blocks of 32
tokens x 32 channels, or the 256 x 256 kernel), with ragged edges and K from a single stage on: the INT8 kernels' bits."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = 'cuda:0'
SHAPES = [(1, 128, 8), (257, 2560, 77), (97, 640, 264),                    # split 1 x 1
          (33, 1024, 4100), (257, 128, 1500),                              # split 1 x 2
          (100, 512, 4104), (333, 128, 2056), (2100, 384, 203), (257, 4096, 3104),      # split 2 x 2
          (257, 4096, 4100), (65, 4096, 11000),                            # split 4 x 2
          (200, 128, 11000), (1000, 128, 2051),                            # 2 x 2
          (257, 384, 6008), (257, 2560, 10999),                            # 2 x 4
          (200, 384, 4104), (1000, 2560, 1031),                            # 4 x 2
          (130, 512, 10999), (1400, 1024, 2056),                           # 4 x 4
          (333, 1024, 11000), (3000, 512, 1501),                           # 4 x 6
          (2100, 128, 3099), (3000, 384, 2056),                            # 8 x 4
          (4098, 256, 2104)]                                               # 256 x 256


@pytest.mark.parametrize('dtype', [torch.bfloat16, torch.float16])
@pytest.mark.parametrize('m,k,n', SHAPES)
def test_every_tile_shape_equals_the_int8_kernels(dtype, m, k, n):
    import quest_amd as quest
    from quest_amd import harness
    g = torch.Generator(device=DEV).manual_seed(m + k + n)
    a = torch.randint(0, 256, (m, k // 2), generator=g, device=DEV, dtype=torch.uint8)
    b = torch.randint(0, 256, (n, k // 2), generator=g, device=DEV, dtype=torch.uint8)
    a[-1], b[-1] = 0x88, 0x88                                              # the largest sum: (-8 + 1/2)^2 K
    a_mul = (torch.rand(m, 1, generator=g, device=DEV) * 0.09 + 0.01).to(dtype)
    b_mul = (torch.rand(n, 1, generator=g, device=DEV) * 0.09 + 0.01).to(dtype)
    a_add = harness.unpack_int4(a).sum(-1, keepdim=True, dtype=torch.int32)
    b_add = harness.unpack_int4(b).sum(-1, keepdim=True, dtype=torch.int32) + k // 2
    ta, tb = quest.int4_to_e2m3_tiles(a), quest.int4_to_e2m3_tiles(b)
    want = quest.fused_matmul_dequantize_int4_int4t_bf16(a, b, a_add, b_add, a_mul, b_mul)
    assert torch.equal(quest.fused_matmul_dequantize_e2m3(ta, tb, a_mul, b_mul, k), want)
    res = (torch.randn(m, n, generator=g, device=DEV) * 30).to(dtype)
    assert torch.equal(quest.fused_matmul_dequantize_e2m3(ta, tb, a_mul, b_mul, k, out=res.clone(), add_to_out=True), res + want)
    if n % 8 == 0 and dtype == torch.bfloat16:                             # (channels: four gates, the four ups of the same outputs, ...)
        gate, up = want.view(m, n // 8, 2, 4).unbind(2)
        glu = (torch.nn.functional.silu(gate) * up).reshape(m, n // 2)
        assert torch.equal(quest.fused_matmul_dequantize_e2m3(ta, tb, a_mul, b_mul, k, swiglu=True), glu)
    if m % 50 == 0 and n % 8 == 0:                                         # sequences of 50 positions, half of the channels rotated
        rot = n // 64 * 32
        ang = torch.rand(50, 16, generator=g, device=DEV) * 6.283
        freqs = torch.stack([torch.cos(ang), torch.sin(ang)], dim=-1).contiguous()
        turned = quest.rope_interleaved_(want.clone().view(-1, 50, n), freqs, rot, 32).view(m, n)
        assert torch.equal(quest.fused_matmul_dequantize_e2m3(ta, tb, a_mul, b_mul, k, rope=(freqs, rot, 32)), turned)


def _operands(m, k, n, dtype):
    import quest_amd as quest
    g = torch.Generator(device=DEV).manual_seed(m + k + n)
    ta, tb = (quest.int4_to_e2m3_tiles(torch.randint(0, 256, (r, k // 2), generator=g, device=DEV, dtype=torch.uint8)) for r in (m, n))
    a_mul, b_mul = ((torch.rand(r, 1, generator=g, device=DEV) * 0.09 + 0.01).to(dtype) for r in (m, n))
    return quest, g, ta, tb, a_mul, b_mul


def _with_bias(quest, ta, tb, a_mul, b_mul, bias, k):
    from quest_amd import _lib
    m, n = a_mul.numel(), b_mul.numel()
    out = torch.empty(m, n, dtype=a_mul.dtype, device=DEV)
    _lib.check(_lib.load().quest_fused_matmul_dequantize_bias_e2m3(
        out.data_ptr(), ta.data_ptr(), tb.data_ptr(), a_mul.data_ptr(), b_mul.data_ptr(), bias.data_ptr(), m, k, n, _lib.DTYPE_CODE[a_mul.dtype],
        torch.cuda.current_stream().cuda_stream), 'bias_e2m3')
    return out


@pytest.mark.parametrize('dtype', [torch.bfloat16, torch.float16])
@pytest.mark.parametrize('m,k,n', SHAPES + [(4100, 256, 2307), (4100, 256, 4099)])
def test_bias_epilogue_of_every_tile_shape(dtype, m, k, n):
    quest, g, ta, tb, a_mul, b_mul = _operands(m, k, n, dtype)
    bias = torch.randn(n, generator=g, device=DEV).to(dtype)
    plain = quest.fused_matmul_dequantize_e2m3(ta, tb, a_mul, b_mul, k)
    assert torch.equal(_with_bias(quest, ta, tb, a_mul, b_mul, bias, k), plain + bias)


def _is_large(m, k, n):
    import ctypes
    from quest_amd import _lib
    plan = (ctypes.c_int * 8)()
    _lib.check(_lib.load().quest_e2m3_gemm_plan(m, k, n, torch.cuda.get_device_properties(0).multi_processor_count, plan), 'plan')
    return list(plan[4:6]) == [256, 256]


@pytest.mark.parametrize('dtype', [torch.bfloat16, torch.float16])
@pytest.mark.parametrize('m,n', [(4100, 2307), (4100, 4099), (4100, 2312), (16900, 520)])
def test_residual_epilogue_of_the_large_tiles(dtype, m, n):
    """Odd widths (element by element), ragged ones and ragged last token tiles."""
    k = 256
    assert _is_large(m, k, n)
    quest, g, ta, tb, a_mul, b_mul = _operands(m, k, n, dtype)
    res = (torch.randn(m, n, generator=g, device=DEV) * 30).to(dtype)
    plain = quest.fused_matmul_dequantize_e2m3(ta, tb, a_mul, b_mul, k)
    assert torch.equal(quest.fused_matmul_dequantize_e2m3(ta, tb, a_mul, b_mul, k, out=res.clone(), add_to_out=True), res + plain)


@pytest.mark.parametrize('dtype', [torch.bfloat16, torch.float16])
@pytest.mark.parametrize('batch,seq,n,rot,head_dim', [(5, 900, 2312, 1536, 32), (5, 900, 2312, 2304, 96), (7, 611, 2088, 192, 64), (100, 41, 2304, 2304, 128)])
def test_rotary_epilogue_of_the_large_tiles(dtype, batch, seq, n, rot, head_dim):
    """Sequences that end inside a tile, narrow heads, a last channel tile that is partly rotated or not at all."""
    m, k = batch * seq, 256
    assert _is_large(m, k, n)
    quest, g, ta, tb, a_mul, b_mul = _operands(m, k, n, dtype)
    ang = torch.rand(seq, head_dim // 2, generator=g, device=DEV) * 6.283
    freqs = torch.stack([torch.cos(ang), torch.sin(ang)], dim=-1).contiguous()
    plain = quest.fused_matmul_dequantize_e2m3(ta, tb, a_mul, b_mul, k)
    want = quest.rope_interleaved_(plain.view(batch, seq, n), freqs, rot, head_dim).view(m, n)
    assert torch.equal(quest.fused_matmul_dequantize_e2m3(ta, tb, a_mul, b_mul, k, rope=(freqs, rot, head_dim)), want)
