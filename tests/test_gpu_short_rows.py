"""Layers on both sides of the rule that sends many tokens with rows of 1536 to 2047 elements to the FP6 kernels: the bits of the
INT8 kernels either way."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = 'cuda:0'


@pytest.mark.parametrize('hadamard', [False, True])
@pytest.mark.parametrize('m,k,n,fp6', [(4097, 1536, 1536, True), (4099, 1664, 1540, True), (4097, 1408, 1536, False), (4097, 1920, 1535, False),
                                       (4096, 1024, 264, True)])
def test_layer_equals_the_int8_path(monkeypatch, m, k, n, fp6, hadamard):
    from quest_amd import harness
    assert harness.prefers_e2m3(m, k, n) == fp6
    g = torch.Generator(device=DEV).manual_seed(m + k + n)
    layer = harness.Linear4bit.from_weight((torch.randn(n, k, device=DEV, generator=g) * 0.02).bfloat16(), None, use_hadamard=hadamard)
    x = torch.randn(m, k, device=DEV, generator=g).bfloat16()
    with torch.no_grad():
        got = layer(x)
        monkeypatch.setattr(harness, 'MATRIX_PATH', 'int8')
        assert torch.equal(got, layer(x))
