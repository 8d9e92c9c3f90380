"""Rows that are not whole 128s on the FP6 path: the activation kernel's tiles with zeros behind the row, the weights' tiles, and layers
against the INT8 kernels; every remainder, every way a row is divided over waves, small and staged tile writes."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = 'cuda:0'


def _tiles_of(x):
    import quest_amd as quest
    from quest_amd import _lib
    m, k = x.shape
    scale = torch.empty(m, 1, dtype=x.dtype, device=DEV)
    tiles = torch.full((quest.e2m3_tiles_bytes(m, (k + 127) // 128 * 128),), 0xAA, dtype=torch.uint8, device=DEV)
    _lib.check(_lib.load().quest_quantize_e2m3_padded(x.data_ptr(), scale.data_ptr(), tiles.data_ptr(), k, m, _lib.DTYPE_CODE[x.dtype],
                                                      torch.cuda.current_stream().cuda_stream), 'quantize_e2m3_padded')
    return scale, tiles


@pytest.mark.parametrize('dtype', [torch.bfloat16, torch.float16])
@pytest.mark.parametrize('m,k', [(5, 32), (33, 160), (70, 224), (64, 480), (40, 992), (37, 1376), (100, 2016), (5, 4064), (9, 4128), (33, 10976),
                                 (3, 32736), (4500, 1056), (2100, 4192), (8300, 736)])
def test_tiles_hold_the_codes_and_zeros_behind_them(dtype, m, k):
    import quest_amd as quest
    from oracle import quest_oracle as qo
    x = torch.randn(m, k, device=DEV, generator=torch.Generator(device=DEV).manual_seed(m + k)).to(dtype)
    x[1, :] = 0
    x[2, 3] = float('nan')
    scale, tiles = _tiles_of(x)
    want_scale, codes, _ = quest.hadamard_quantize_int4(x, hadamard_scale=0.)
    assert torch.equal(scale.view(torch.int16), want_scale.view(torch.int16))
    values = qo.e2m3_tiles_decode(tiles.cpu(), m, (k + 127) // 128 * 128)
    assert torch.equal(values[:, :k], qo.unpack_int4(codes.cpu()).double() + 0.5)
    assert bool((values[:, k:] == 0).all())


@pytest.mark.parametrize('rows,k', [(1, 32), (33, 96), (100, 1376), (64, 2016), (5, 128)])
def test_weight_tiles(rows, k):
    import quest_amd as quest
    from oracle import quest_oracle as qo
    packed = torch.randint(0, 256, (rows, k // 2), dtype=torch.uint8, device=DEV, generator=torch.Generator(device=DEV).manual_seed(k))
    values = qo.e2m3_tiles_decode(quest.api.int4_to_e2m3_tiles_padded(packed).cpu(), rows, (k + 127) // 128 * 128)
    assert torch.equal(values[:, :k], qo.unpack_int4(packed.cpu()).double() + 0.5) and bool((values[:, k:] == 0).all())


@pytest.mark.parametrize('dtype', [torch.bfloat16, torch.float16])
@pytest.mark.parametrize('m,k,n,bias', [(333, 1376, 4096, False), (100, 2016, 1031, True), (60, 4064, 2048, False), (1000, 1056, 2560, True), (4200, 1888, 2056, False)])
def test_layers_equal_the_int8_kernels(dtype, m, k, n, bias):
    from quest_amd import harness
    g = torch.Generator(device=DEV).manual_seed(m + k + n)
    layer = harness.Linear4bit.from_weight((torch.randn(n, k, device=DEV, generator=g) * .02).to(dtype), torch.randn(n, device=DEV, generator=g).to(dtype) if bias else None)
    assert harness.prefers_e2m3(m, harness.tiles_k(k, False), n) and layer._kept_tiles() is not None and layer.readable_tiles() is None
    x = torch.randn(m, k, device=DEV, generator=g).to(dtype)
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CUDA]) as prof:
        got = layer(x)
        torch.cuda.synchronize()
    assert any('e2m3' in e.key and 'gemm' in e.key for e in prof.key_averages())
    want = harness.linear_forward(x, layer.w_int_packed, layer.w_scale, layer.w_add)
    want = want if layer.bias is None else want + layer.bias
    assert torch.equal(got, want)
    layer.w_int_packed.zero_()                                       # written by hand: the packed codes serve until the tiles are laid out again
    assert layer._kept_tiles() is None
    assert torch.equal(layer(x), harness.linear_forward(x, layer.w_int_packed, layer.w_scale, layer.w_add) + (0 if layer.bias is None else layer.bias))


def _kernels(call):
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CUDA]) as prof:
        call()
        torch.cuda.synchronize()
    return [e.key for e in prof.key_averages()]


def test_rows_that_are_too_long_for_the_quantiser_stay_native(monkeypatch):
    """Packed codes, and no tiles that nothing could read: the call is not left to the Python statement."""
    from quest_amd import harness
    g = torch.Generator(device=DEV).manual_seed(1)
    layer = harness.Linear4bit.from_weight((torch.randn(96, 33056, device=DEV, generator=g) * .02).half())
    x = torch.randn(600, 33056, device=DEV, generator=g).half()
    want = harness.linear_forward(x, layer.w_int_packed, layer.w_scale, layer.w_add)
    assert layer._tiles is None

    def declined(*_, **__):
        raise AssertionError('the native call declined')
    monkeypatch.setattr(harness, 'linear_forward', declined)
    assert torch.equal(layer(x), want)
    layer._tiles = (torch.zeros(1), layer.w_int_packed, layer.w_int_packed.data_ptr(), layer.w_int_packed._version)      # (as of a loaded object)
    assert torch.equal(layer(x), want)


@pytest.mark.parametrize('m,k,n,tiles', [(49, 3104, 4096, False), (56, 4064, 1024, False), (57, 3104, 1024, True), (50, 4128, 1024, True), (50, 2272, 16416, True), (52, 1568, 1024, True),
                                           (300, 1376, 3319, False), (300, 1376, 3320, True), (300, 1376, 1031, True), (500, 2016, 2052, False), (500, 2080, 2052, True),
                                           (1000, 1056, 2201, True), (1000, 1056, 2199, False)])
def test_which_ragged_layers_take_tiles(m, k, n, tiles):
    from quest_amd import harness
    g = torch.Generator(device=DEV).manual_seed(m + k + n)
    layer = harness.Linear4bit.from_weight((torch.randn(n, k, device=DEV, generator=g) * .02).half())
    x, got = torch.randn(m, k, device=DEV, generator=g).half(), []
    assert any('e2m3' in name for name in _kernels(lambda: got.append(layer(x)))) == tiles
    assert torch.equal(got[0], harness.linear_forward(x, layer.w_int_packed, layer.w_scale, layer.w_add))
