"""`Linear4bit` used as a module in a user's program: derivatives of its bias, buffers that are no longer plain buffers."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = 'cuda:0'


def layer_and_input(m=70, k=256, n=264, bias=True, dtype=torch.bfloat16, seed=31):
    from quest_amd import harness
    g = torch.Generator(device=DEV).manual_seed(seed)
    w = (torch.randn(n, k, device=DEV, generator=g) * 0.02).to(dtype)
    b = torch.randn(n, device=DEV, generator=g).to(dtype) if bias else None
    return harness.Linear4bit.from_weight(w, b, use_hadamard=True), torch.randn(m, k, device=DEV, generator=g).to(dtype)


@pytest.mark.parametrize('m', [3, 70])
def test_bias_gradient_and_tangent(m):
    layer, x = layer_and_input(m)
    want = layer(x)
    layer.bias.requires_grad_(True)
    y = layer(x)
    assert torch.equal(y, want)
    y.sum().backward()
    assert torch.equal(layer.bias.grad, torch.full_like(layer.bias, float(m)))       # m ones: exact in bf16
    with torch.no_grad():
        assert not layer(x).requires_grad
    layer.bias.requires_grad_(False)
    import torch.autograd.forward_ad as fw
    from torch.func import functional_call
    with fw.dual_level():
        t = torch.randn_like(layer.bias)
        out = functional_call(layer, {'bias': fw.make_dual(layer.bias.detach(), t)}, (x,))
        assert torch.equal(fw.unpack_dual(out).tangent, t.expand(m, -1))


def test_sparse_metadata_is_refused_and_other_holders_of_the_buffers_work():
    layer, x = layer_and_input()
    want = layer(x)
    layer.w_meta_e = torch.zeros(1, dtype=torch.uint8, device=DEV)
    with pytest.raises(NotImplementedError):
        layer(x)
    layer.w_meta_e = None
    packed = layer.w_int_packed
    del layer.w_int_packed
    layer.w_int_packed = torch.nn.Parameter(packed, requires_grad=False)
    assert torch.equal(layer(x), want)
