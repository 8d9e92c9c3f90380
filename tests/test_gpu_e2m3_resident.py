"""The FP6 GEMM that keeps a channel tile's weights in LDS, against the INT8 kernels: every epilogue at ragged edges, the shortest and
longest rows (an odd number of 128-k stages among them), whole tiles and runs over several tiles per workgroup, idle waves and XCDs."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = 'cuda:0'
# (the gated epilogue takes outputs in whole 16-byte pieces too: channels in whole sixteens)
SHAPES = [(800, 512, 11008), (600, 640, 11024), (3000, 1024, 2064), (5503, 1664, 2064), (8200, 768, 3088), (2111, 1536, 5648), (16500, 1152, 6160)]
EIGHTS = [(3000, 1024, 2056), (5503, 1664, 2056), (8200, 768, 3080)]        # ... and these run the gated epilogue on other kernels


def _plan(m, k, n):
    from quest_amd import _lib
    plan = (ctypes.c_int * 8)()
    _lib.check(_lib.load().quest_e2m3_gemm_plan(m, k, n, torch.cuda.get_device_properties(0).multi_processor_count, plan), 'plan')
    return list(plan)


@pytest.mark.parametrize('dtype', [torch.bfloat16, torch.float16])
@pytest.mark.parametrize('m,k,n', SHAPES + EIGHTS)
def test_every_epilogue_equals_the_int8_kernels(dtype, m, k, n):
    import quest_amd as quest
    from quest_amd import _lib, harness
    assert _plan(m, k, n)[4:] == [64, 128, 1, k]
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
    # channels: four gates, the four ups of the same outputs, ...; the INT8 kernels' gated epilogue has the same arithmetic
    glu = quest.fused_matmul_dequantize_swiglu_int4_int4t(a, b, a_add, b_add, a_mul, b_mul)
    assert torch.equal(quest.fused_matmul_dequantize_e2m3(ta, tb, a_mul, b_mul, k, swiglu=True), glu)
    if dtype == torch.bfloat16:
        gate, up = want.view(m, n // 8, 2, 4).unbind(2)
        assert torch.equal(glu, (torch.nn.functional.silu(gate) * up).reshape(m, n // 2))
    for seq, head_dim in ((37, 32), (max(32, m // 7), 96)):                # heads that a channel tile cuts, sequences that a block cuts
        rows = m // seq * seq
        rot = n // 2 // head_dim * head_dim
        ang = torch.rand(seq, head_dim // 2, generator=g, device=DEV) * 6.283
        freqs = torch.stack([torch.cos(ang), torch.sin(ang)], dim=-1).contiguous()
        turned = quest.rope_interleaved_(want[:rows].clone().view(-1, seq, n), freqs, rot, head_dim).view(rows, n)
        assert torch.equal(quest.fused_matmul_dequantize_e2m3(quest.int4_to_e2m3_tiles(a[:rows].contiguous()), tb, a_mul[:rows], b_mul, k, rope=(freqs, rot, head_dim)), turned)


def test_the_shapes_take_both_kinds_of_plan():
    """One or several workgroups per channel tile, and even runs over an XCD's tiles; every shape also gated."""
    shared = [_plan(*s)[2] for s in SHAPES]
    assert 0 in shared and 1 < max(shared) and all(n % 16 == 0 for _, _, n in SHAPES)


def test_scales_at_the_edge_of_the_range():
    """The sums come out of the products doubled and the scales' product is halved first: no overflow or underflow that the INT8 kernels
    do not have."""
    import quest_amd as quest
    from quest_amd import harness
    m, k, n = 3000, 1024, 2056
    assert _plan(m, k, n)[4:] == [64, 128, 1, k]
    g = torch.Generator(device=DEV).manual_seed(1)
    a = torch.randint(0, 256, (m, k // 2), generator=g, device=DEV, dtype=torch.uint8)
    b = torch.randint(0, 256, (n, k // 2), generator=g, device=DEV, dtype=torch.uint8)
    a_mul = torch.exp2(torch.randint(-130, 128, (m, 1), generator=g, device=DEV).double()).bfloat16()
    b_mul = torch.exp2(torch.randint(-130, 128, (n, 1), generator=g, device=DEV).double()).bfloat16() * 1.2890625
    a_mul[:4, 0] = torch.tensor([0., float('inf'), float('nan'), 3.3e38], device=DEV)
    a_add = harness.unpack_int4(a).sum(-1, keepdim=True, dtype=torch.int32)
    b_add = harness.unpack_int4(b).sum(-1, keepdim=True, dtype=torch.int32) + k // 2
    want = quest.fused_matmul_dequantize_int4_int4t_bf16(a, b, a_add, b_add, a_mul, b_mul)
    got = quest.fused_matmul_dequantize_e2m3(quest.int4_to_e2m3_tiles(a), quest.int4_to_e2m3_tiles(b), a_mul, b_mul, k)
    assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got.nan_to_num(0.), want.nan_to_num(0.))
