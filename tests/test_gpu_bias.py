"""A layer's bias in the GEMM's epilogue: the bits of the layer without it plus torch's addition, for every kernel of the dispatch,
edge tiles and biases that start at any element of a buffer."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = 'cuda:0'


@pytest.mark.parametrize('dtype', [torch.bfloat16, torch.float16])
@pytest.mark.parametrize('path', ['int8', 'fp6'])
@pytest.mark.parametrize('offset', [0, 1])
@pytest.mark.parametrize('m,k,n', [(1, 1376, 24), (17, 128, 4099), (64, 256, 264), (70, 1376, 77), (333, 512, 1032), (1000, 2560, 2560), (1700, 288, 3003),
                                   (2100, 4096, 4104)])
def test_bias_is_added_to_the_rounded_product(monkeypatch, m, k, n, offset, path, dtype):
    from quest_amd import harness
    monkeypatch.setattr(harness, 'MATRIX_PATH', path)
    g = torch.Generator(device=DEV).manual_seed(m + n)
    x = torch.randn(m, k, device=DEV, generator=g).to(dtype)
    layer = harness.Linear4bit.from_weight((torch.randn(n, k, device=DEV, generator=g) * 0.02).to(dtype))
    bias = torch.randn(n + offset, device=DEV, generator=g).to(dtype)[offset:]
    want = layer(x) + bias
    layer.bias = torch.nn.Parameter(bias, requires_grad=False)
    assert torch.equal(layer(x), want)
