"""The FP6 GEMM's 128 x 96 tiles, whose waves share K by pairs, against the INT8 kernels: an even and an odd number
of stages, ragged edges, every epilogue."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = 'cuda:0'
SHAPES = [(1000, 1152, 2560), (500, 1280, 4100), (1400, 1664, 2051), (333, 1792, 6008), (130, 1152, 10999), (200, 2560, 11008), (333, 11008, 6008)]


def _plan(m, k, n):
    from quest_amd import _lib
    plan = (ctypes.c_int * 8)()
    _lib.check(_lib.load().quest_e2m3_gemm_plan(m, k, n, torch.cuda.get_device_properties(0).multi_processor_count, plan), 'plan')
    return list(plan)


@pytest.mark.parametrize('dtype', [torch.bfloat16, torch.float16])
@pytest.mark.parametrize('m,k,n', SHAPES)
def test_every_epilogue_equals_the_int8_kernels(dtype, m, k, n):
    import quest_amd as quest
    from quest_amd import _lib, harness
    assert _plan(m, k, n)[4:] == [128, 96, 7, 128]
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
    guard = torch.full((m + 1, n), 7., dtype=dtype, device=DEV)            # (nothing is written past the last row)
    got = quest.fused_matmul_dequantize_e2m3(ta, tb, a_mul, b_mul, k, out=guard[:m])
    assert torch.equal(got, want) and bool((guard[m] == 7.).all())
    res = (torch.randn(m, n, generator=g, device=DEV) * 30).to(dtype)
    assert torch.equal(quest.fused_matmul_dequantize_e2m3(ta, tb, a_mul, b_mul, k, out=res.clone(), add_to_out=True), res + want)
    bias = torch.randn(n, generator=g, device=DEV).to(dtype)
    out = torch.empty(m, n, dtype=dtype, device=DEV)
    _lib.check(_lib.load().quest_fused_matmul_dequantize_bias_e2m3(
        out.data_ptr(), ta.data_ptr(), tb.data_ptr(), a_mul.data_ptr(), b_mul.data_ptr(), bias.data_ptr(), m, k, n, _lib.DTYPE_CODE[dtype],
        torch.cuda.current_stream().cuda_stream), 'bias_e2m3')
    assert torch.equal(out, want + bias)
    if n % 8:
        return
    glu = quest.fused_matmul_dequantize_swiglu_int4_int4t(a, b, a_add, b_add, a_mul, b_mul)
    assert torch.equal(quest.fused_matmul_dequantize_e2m3(ta, tb, a_mul, b_mul, k, swiglu=True), glu)
    for seq, head_dim in ((37, 32), (max(32, m // 7), 96)):                # heads that a channel tile cuts, sequences that a block cuts
        rows, rot = m // seq * seq, n // 2 // head_dim * head_dim
        ang = torch.rand(seq, head_dim // 2, generator=g, device=DEV) * 6.283
        freqs = torch.stack([torch.cos(ang), torch.sin(ang)], dim=-1).contiguous()
        turned = quest.rope_interleaved_(want[:rows].clone().view(-1, seq, n), freqs, rot, head_dim).view(rows, n)
        assert torch.equal(quest.fused_matmul_dequantize_e2m3(quest.int4_to_e2m3_tiles(a[:rows].contiguous()), tb, a_mul[:rows], b_mul, k, rope=(freqs, rot, head_dim)), turned)
