"""The activation kernel that reads ahead for the GEMM behind it: the outputs of the entry points without, whatever it reads -- no piece,
fewer pieces than XCDs, pieces of one chunk, whole weights -- for every producer, both code forms, every way a row is divided over waves."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = 'cuda:0'
EPS = 1e-5
NEXT = [(0, 0, 0), (1, 16, 16), (7, 4096, 48), (8, 1536, 1536), (129, 24576, 8000)]                  # (pieces, pitch, bytes of each)


def _run(producer, x, branch, weight, tiles, had_scale, next_):
    from quest_amd import _lib
    import quest_amd as quest
    m, k = x.size(0), x.size(1) // (2 if producer == 2 else 1)
    scale = torch.empty(m, 1, dtype=x.dtype, device=DEV)
    packed, row_sum = torch.empty(m, k // 2, dtype=torch.uint8, device=DEV), torch.empty(m, 1, dtype=torch.int32, device=DEV)
    t = torch.zeros(quest.e2m3_tiles_bytes(m, k), dtype=torch.uint8, device=DEV)
    pieces, pitch, each = next_
    memory = torch.zeros(max(16, pieces * pitch), dtype=torch.uint8, device=DEV)
    a = _lib.Activation(producer, x.data_ptr(), 0 if branch is None else branch.data_ptr(), weight.data_ptr(), EPS, scale.data_ptr(),
                        0 if tiles else packed.data_ptr(), 0 if tiles else row_sum.data_ptr(), t.data_ptr() if tiles else 0, k, m, had_scale,
                        _lib.DTYPE_CODE[x.dtype], memory.data_ptr() if pieces else 0, pitch, each, pieces)
    _lib.check(_lib.load().quest_activation_before_gemm(ctypes.byref(a), torch.cuda.current_stream().cuda_stream), 'activation_before_gemm')
    return (scale, t) if tiles else (scale, packed, row_sum)


def _codes(tiles, m, k):
    """The bytes of m rows' codes: a fragment is 64 lanes (row, half of the 64 elements) of sixteen bytes and then of eight, and rows past m hold anything."""
    t = tiles.view(-1, k // 64, 1536)
    heads, tails = (part.reshape(*t.shape[:2], 2, 32, -1) for part in (t[..., :1024], t[..., 1024:]))
    rows = torch.cat((heads, tails), -1).permute(0, 3, 1, 2, 4).reshape(t.size(0) * 32, -1)[:m]
    assert rows.shape == (m, k // 4 * 3)
    return rows


@pytest.mark.parametrize('dtype', [torch.bfloat16, torch.float16])
@pytest.mark.parametrize('hadamard', [True, False])
@pytest.mark.parametrize('tiles', [False, True])
@pytest.mark.parametrize('producer', ['none', 'norm', 'add_norm', 'silu'])
@pytest.mark.parametrize('m,k', [(37, 1024), (5, 1920), (100, 2816), (9, 4224), (33, 11008), (4200, 1024), (3, 512), (2, 12416)])
def test_outputs_are_those_of_the_entry_points_without(tiles, producer, m, k, hadamard, dtype):
    import quest_amd as quest
    from quest_amd import harness
    g = torch.Generator(device=DEV).manual_seed(m + k)
    x, other = (torch.randn(m, k * (2 if producer == 'silu' else 1), device=DEV, generator=g).to(dtype) for _ in range(2))
    weight = torch.rand(k, device=DEV, generator=g).to(dtype)
    branch = other if producer == 'add_norm' else None
    kind = {'none': 0, 'norm': 1, 'add_norm': 1, 'silu': 2}[producer]
    had_scale = harness.HADAMARD_ENTRY if hadamard else 0.
    plain = x if branch is None else x + branch
    form = 'e2m3' if tiles else 'int4'
    want = (getattr(quest, f'hadamard_quantize_{form}')(plain, hadamard_scale=had_scale) if kind == 0
            else getattr(quest, f'rmsnorm_hadamard_quantize_{form}')(plain, weight, EPS, hadamard_scale=had_scale) if kind == 1
            else getattr(quest, f'silu_mul_hadamard_quantize_{form}')(plain, hadamard_scale=had_scale))
    if tiles:
        want = want[0], _codes(want[1], m, k)
    for next_ in [NEXT[0], *(NEXT[1:] if (m, k) in ((37, 1024), (4200, 1024)) else NEXT[-1:])]:
        mine = x.clone()
        got = _run(kind, mine, branch, weight, tiles, had_scale, next_)
        assert torch.equal(mine, plain)                              # (with a branch: replaced by the sum)
        if tiles:
            got = got[0], _codes(got[1], m, k)
        for a, b in zip(got, want):
            assert torch.equal(a.view(torch.uint8), b.view(torch.uint8))


def test_what_it_refuses():
    from quest_amd import _lib
    lib = _lib.load()
    x = torch.zeros(4, 1024, dtype=torch.bfloat16, device=DEV)
    s = torch.zeros(4, 1, dtype=torch.bfloat16, device=DEV)
    t = torch.zeros(24576 * 4, dtype=torch.uint8, device=DEV)

    def status(**change):
        a = _lib.Activation(0, x.data_ptr(), 0, 0, EPS, s.data_ptr(), 0, 0, t.data_ptr(), 1024, 4, .08837890625, 0, 0, 0, 0, 0)
        for name, value in change.items():
            setattr(a, name, value)
        return lib.quest_activation_before_gemm(ctypes.byref(a), torch.cuda.current_stream().cuda_stream)
    assert status() == 0 and lib.quest_activation_before_gemm(None, None) == -1
    assert status(tiles=0) == -1 and status(producer=1) == -1 and status(size_k=1000) == -2 and status(dtype=7) == -3
    assert status(producer=3) != 0 and status(branch=x.data_ptr()) != 0 and status(had_scale=.1) != 0 and status(x=x.data_ptr() + 2) != 0
