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


@pytest.mark.parametrize('m', [3, 40, 96, 200, 1000])
@pytest.mark.parametrize('direct', [False, True])
def test_scales_at_an_odd_element(m, direct):
    """A slice of a longer scale vector: only some kernels read it, and a layer finds them at every size."""
    from quest_amd import harness
    layer, x = layer_and_input(m, 2048, 1024, bias=False)
    want = layer(x)
    layer.w_scale = torch.cat([layer.w_scale[:1], layer.w_scale])[1:]
    assert layer.w_scale.data_ptr() % 4 == 2 and layer.tiles_for(m) is None
    if direct:
        got = harness.linear_forward(x, layer.w_int_packed, layer.w_scale, layer.w_add, use_hadamard=True, w_tiles=layer.w_tiles())
    else:
        got = layer(x)
    assert torch.equal(got, want)
    odd = torch.empty(m + 1, 1, dtype=x.dtype, device=DEV)[1:]
    got = harness.linear_forward(x, layer.w_int_packed, layer.w_scale, layer.w_add, use_hadamard=True, w_tiles=layer.w_tiles(), _a_scale=odd)
    assert torch.equal(got, want)


def test_more_rows_than_tiles_can_hold():
    """2^21 + 32 channels: no tiles are laid out, and the packed codes serve."""
    from quest_amd import harness
    n, k, m = 2 ** 21 + 32, 512, 70
    g = torch.Generator(device=DEV).manual_seed(5)
    layer = harness.Linear4bit.empty(k, n, device=DEV, dtype=torch.bfloat16, use_hadamard=True)
    layer.w_int_packed.random_(0, 256, generator=g)
    layer.w_scale.fill_(0.01)
    layer.lay_out_tiles()
    x = torch.randn(m, k, device=DEV, generator=g).bfloat16()
    y = layer(x)
    assert torch.equal(y[:, -40:], harness.linear_forward(x, layer.w_int_packed[-40:], layer.w_scale[-40:], layer.w_add[-40:], use_hadamard=True))
