"""A layer on a few tokens in one launch against the activation kernel and the GEMM one after the other: every way a row is divided
over waves (rows of 5 to 96 blocks), the most tokens of each, ragged channels, more tiles than workgroups, degenerate rows, a bias."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = 'cuda:0'
WHOLE = [(1, 4096, 4096), (8, 4096, 4100), (16, 1024, 1024), (16, 640, 300), (7, 2816, 1031), (3, 768, 17), (4, 8192, 2048), (2, 11008, 4096),
         (2, 12288, 333), (2, 4224, 5000), (1, 11008, 22016), (16, 1408, 6000), (1, 1024, 1), (16, 2048, 9000)]
RAGGED = [(1, 1376, 4096), (8, 4064, 1000), (2, 10976, 640), (4, 5472, 2000), (11, 672, 50)]          # whole 32s, without the transform
REFUSED = [(9, 4096, 512), (17, 1024, 512), (5, 8192, 512), (3, 11008, 512), (1, 512, 512), (1, 12416, 512)]


def _operands(m, k, n, dtype):
    g = torch.Generator(device=DEV).manual_seed(m * k + n)
    x = torch.randn(m, k, device=DEV, generator=g).to(dtype)
    if m > 3:
        x[1], x[2, 5], x[3, 7] = 0, float('nan'), float('inf')
    w = torch.randint(0, 256, (n, k // 2), dtype=torch.uint8, device=DEV, generator=g)
    from quest_amd import harness
    add = harness.unpack_int4(w).sum(-1, keepdim=True, dtype=torch.int32) + k // 2
    return x, w, add, (torch.rand(n, 1, device=DEV, generator=g) * .1).to(dtype), torch.randn(n, device=DEV, generator=g).to(dtype)


def _one_launch(x, w, add, scale, bias, had_scale):
    from quest_amd import _lib
    m, n = x.size(0), w.size(0)
    out = torch.full((m + 1, n), 7., dtype=x.dtype, device=DEV)
    rc = _lib.load().quest_linear_few_tokens(out.data_ptr(), x.data_ptr(), w.data_ptr(), add.data_ptr(), scale.data_ptr(), 0 if bias is None else bias.data_ptr(),
                                             m, x.size(1), n, had_scale, _lib.DTYPE_CODE[x.dtype], torch.cuda.current_stream().cuda_stream)
    assert bool((out[m] == 7.).all())                                      # nothing is written past the last row
    return rc, out[:m]


@pytest.mark.parametrize('dtype', [torch.bfloat16, torch.float16])
@pytest.mark.parametrize('hadamard,m,k,n', [(h, *s) for s in WHOLE for h in (True, False)] + [(False, *s) for s in RAGGED])
def test_equals_the_two_launches(dtype, hadamard, m, k, n):
    import quest_amd as quest
    from quest_amd import harness
    had_scale = harness.HADAMARD_ENTRY if hadamard else 0.
    x, w, add, scale, bias = _operands(m, k, n, dtype)
    a_scale, codes, row_sum = quest.hadamard_quantize_int4(x, hadamard_scale=had_scale)
    want = quest.fused_matmul_dequantize_int4_int4t_bf16(mat_a=codes, mat_b=w, vec_a_add=row_sum, vec_b_add=add, vec_a_mul=a_scale, vec_b_mul=scale)
    for b in (None, bias):
        rc, got = _one_launch(x, w, add, scale, b, had_scale)
        assert rc == 0
        expected = want if b is None else want + b
        same = (got == expected) | (got.isnan() & expected.isnan())
        assert bool(same.all())


@pytest.mark.parametrize('m,k,n', REFUSED)
def test_other_sizes_take_the_two_launches(m, k, n):
    from quest_amd import harness
    x, w, add, scale, bias = _operands(m, k, n, torch.bfloat16)
    rc, out = _one_launch(x, w, add, scale, bias, harness.HADAMARD_ENTRY)
    assert rc != 0 and bool((out == 7.).all())
    layer = harness.linear_forward(x, w, scale, add, use_hadamard=True)
    assert layer.shape == (m, n)


def test_graph_replays():
    from quest_amd import harness
    x, w, add, scale, bias = _operands(2, 4096, 11008, torch.float16)
    eager = harness.linear_forward(x, w, scale, add, use_hadamard=True)
    stream, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        out = harness.linear_forward(x, w, scale, add, use_hadamard=True)
    for _ in range(3):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, eager)


@pytest.mark.parametrize('m,k', [(8, 4096), (16, 1024), (40, 1024)])
def test_output_in_the_place_of_the_input(m, k):
    from quest_amd import harness
    x, w, add, scale, _ = _operands(m, k, k, torch.bfloat16)
    x = torch.randn(m, k, device=DEV).bfloat16()
    for tiles in (None, harness.weight_tiles(w)):
        want = harness.linear_forward(x, w, scale, add, use_hadamard=True, w_tiles=tiles)
        for _ in range(5):
            both = x.clone()
            got = harness.linear_forward(both, w, scale, add, use_hadamard=True, w_tiles=tiles, out=both)
            assert got is both and torch.equal(got, want)
