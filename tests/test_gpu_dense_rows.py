"""Norm and dense head of a few rows against fp64: each output is one rounding to the dtype away from a sum whose fp32
accumulation error is below K * 2^-24 of the sum of magnitudes."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = 'cuda:0'
ULP = {torch.bfloat16: 2. ** -8, torch.float16: 2. ** -11}


@pytest.mark.parametrize('dtype', [torch.bfloat16, torch.float16])
@pytest.mark.parametrize('m,k,n', [(1, 64, 5), (16, 1024, 320), (17, 576, 33), (32, 2560, 1000), (33, 1088, 40), (64, 1024, 3200)])
def test_dense_rows(dtype, m, k, n):
    from quest_amd import _lib
    g = torch.Generator(device=DEV).manual_seed(m + n)
    x, w = torch.randn(m, k, device=DEV, generator=g).to(dtype), torch.randn(n, k, device=DEV, generator=g).to(dtype)
    out = torch.full((m + 1, n), 7., dtype=dtype, device=DEV)
    _lib.check(_lib.load().quest_dense_rows(out.data_ptr(), x.data_ptr(), w.data_ptr(), m, k, n, _lib.DTYPE_CODE[dtype],
                                            torch.cuda.current_stream().cuda_stream), 'dense_rows')
    want, mag = x.double() @ w.double().t(), x.double().abs() @ w.double().abs().t()
    assert ((out[:m].double() - want).abs() <= want.abs() * ULP[dtype] + mag * k * 2. ** -24).all()
    assert (out[m] == 7.).all()


@pytest.mark.parametrize('with_branch', [False, True])
@pytest.mark.parametrize('b,t,c', [(1, 1, 64), (3, 5, 1024), (64, 2, 2560)])
def test_last_logits(with_branch, b, t, c):
    """Against the module's own norm and head on the last positions: a logit is rounded once (2^-8 of itself at most); the
    two norms differ by one unit in the last place on a few elements (fp32 order of the mean), which adds less than that."""
    from quest_amd import _lib, llama
    g = torch.Generator(device=DEV).manual_seed(b)
    x, branch = (torch.randn(b, t, c, device=DEV, generator=g).bfloat16() for _ in range(2))
    norm = llama.RMSNorm(c).to(DEV).bfloat16()
    norm.weight.data.uniform_(0.5, 1.5)
    head = torch.randn(77, c, device=DEV, generator=g).bfloat16()
    with torch.no_grad():
        got = _lib.host.last_logits(x, branch if with_branch else None, norm.weight, norm.eps, head)
        want = norm((x + branch if with_branch else x)[:, -1:]).double() @ head.double().t()
    assert got.shape == (b, 1, 77)
    assert (got.double() - want).norm() <= 2. ** -7 * want.norm()
