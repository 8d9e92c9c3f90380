"""Rows of whole 32s that are not whole 128s, without the transform: one order of the sum of squares, and so one result of a row, in every call -- whatever
the number of rows beside it, on packed codes and on tiles, natively and in the Python statement of the call."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = 'cuda:0'


def _rows_between_two_scales(count, k, dtype):
    """The `count` of 65536 Gaussian rows (16384 long ones) whose scale is nearest to the middle between two values of the dtype, nearest first: sums of
    squares in two orders round to different scales on some of them."""
    from oracle import quest_oracle as qo
    g = torch.Generator(device=DEV).manual_seed(k)
    rows, off = [], []
    for _ in range(16 if k <= 16384 else 4):
        x = torch.randn(4096, k, device=DEV, generator=g).to(dtype)
        s = x.double().square().mean(-1).sqrt() * qo.GAUSS_INT4_STEP + qo.SCALE_EPS               # the rule's scale in 64 bits
        ulp = torch.exp2(torch.floor(torch.log2(s)) - (10 if dtype == torch.float16 else 7))
        rows.append(x)
        off.append(((s / ulp).frac() - 0.5).abs())
    rows, off = torch.cat(rows), torch.cat(off)
    return rows[off.argsort()[:count]].contiguous()


def _tiles(x):
    import quest_amd as quest
    from quest_amd import _lib
    m, k = x.shape
    scale, tiles = torch.empty(m, 1, dtype=x.dtype, device=DEV), torch.zeros(quest.e2m3_tiles_bytes(m, (k + 127) // 128 * 128), dtype=torch.uint8, device=DEV)
    _lib.check(_lib.load().quest_quantize_e2m3_padded(x.data_ptr(), scale.data_ptr(), tiles.data_ptr(), k, m, _lib.DTYPE_CODE[x.dtype],
                                                      torch.cuda.current_stream().cuda_stream), 'quantize_e2m3_padded')
    return scale, tiles


@pytest.mark.parametrize('dtype', [torch.bfloat16, torch.float16])
@pytest.mark.parametrize('k', [32, 96, 160, 480, 992, 1376, 2016, 4064, 4128, 10976, 16416, 32736])
def test_codes_and_tiles_have_the_same_scales(dtype, k):
    import quest_amd as quest
    from oracle import quest_oracle as qo
    x = _rows_between_two_scales(333, k, dtype)
    x[1], x[2, 5], x[3, 7] = 0, float('nan'), float('inf')
    kept = torch.full((334, k), 7., dtype=dtype, device=DEV)
    scale, codes, row_sum = quest.hadamard_quantize_int4(x, hadamard_scale=0., x_had=kept[:333])
    assert torch.equal(kept[:333].view(torch.int16), x.view(torch.int16)) and bool((kept[333] == 7.).all())
    into = torch.full((333 * k // 2 + 20,), 0xAA, dtype=torch.uint8, device=DEV)              # codes that start four bytes into an allocation
    quest.hadamard_quantize_int4(x, x_int_packed=into[4:-16].view(333, k // 2), hadamard_scale=0.)
    assert torch.equal(into[4:-16].view(333, k // 2), codes) and bool((into[:4] == 0xAA).all()) and bool((into[-16:] == 0xAA).all())
    again, tiles = _tiles(x)
    assert torch.equal(scale.view(torch.int16), again.view(torch.int16))
    q = qo.unpack_int4(codes.cpu())
    assert torch.equal(row_sum.cpu().flatten(), q.sum(-1, dtype=torch.int32))
    assert torch.equal(qo.e2m3_tiles_decode(tiles.cpu(), 333, (k + 127) // 128 * 128)[:, :k], q.double() + 0.5)
    # ... and the codes are the quantiser's for that scale (the degenerate rows aside)
    want = torch.empty(329, k // 2, dtype=torch.uint8)
    qo.quantize_int4(x[4:].cpu(), scale[4:].cpu(), None, want, torch.empty(329, 1, dtype=torch.int32), False)
    assert torch.equal(codes[4:].cpu(), want)


@pytest.mark.parametrize('dtype', [torch.bfloat16, torch.float16])
@pytest.mark.parametrize('k,n', [(1376, 1000), (672, 4096), (4064, 512), (10976, 264)])
def test_a_row_has_one_result(monkeypatch, dtype, k, n):
    from quest_amd import harness
    import quest_amd as quest
    g = torch.Generator(device=DEV).manual_seed(k)
    layer = harness.Linear4bit.from_weight((torch.randn(n, k, device=DEV, generator=g) * .02).to(dtype))
    x = _rows_between_two_scales(600, k, dtype)
    with torch.no_grad():
        want = layer(x)
        for m in (1, 2, 4, 8, 11, 16, 20, 40, 60, 100, 333):
            assert torch.equal(layer(x[:m]), want[:m]), m
        scratch = torch.empty(600, 1, dtype=dtype, device=DEV)             # given scratch: the Python statement
        assert torch.equal(harness.linear_forward(x, layer.w_int_packed, layer.w_scale, layer.w_add, _a_scale=scratch), want)
        scale, codes, row_sum = quest.hadamard_quantize_int4(x, hadamard_scale=0.)
        assert torch.equal(layer.forward_quantized(scale, codes, row_sum), want)
        monkeypatch.setattr(harness, 'MATRIX_PATH', 'int8')
        for m in (1, 8, 60, 333, 600):
            assert torch.equal(layer(x[:m]), want[:m]), m
