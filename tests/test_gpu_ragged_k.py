"""GEMM on rows that are not whole stages of a kernel (K % 32 == 0 only): the int32 matrix against the exact product, for
every kernel of the dispatch."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = 'cuda:0'


@pytest.mark.parametrize('m,n', [(1, 24), (17, 40), (64, 4100), (65, 72), (130, 3000), (1000, 4096), (2300, 1032), (3000, 9000)])
@pytest.mark.parametrize('k', [32, 96, 128, 160, 224, 288, 416, 1376])
def test_matmul_int32_exact(m, k, n):
    """Extreme and random codes; the bytes after the last row are another operand's, so a read past a row's end shows."""
    import quest_amd as quest
    from quest_amd import harness
    g = torch.Generator(device=DEV).manual_seed(m + k + n)
    pool = torch.randint(0, 256, ((m + n + 4) * k // 2,), dtype=torch.uint8, device=DEV, generator=g)
    a, b = pool[:m * k // 2].view(m, k // 2), pool[m * k // 2:(m + n) * k // 2].view(n, k // 2)
    a[0], b[-1] = 0x88, 0x88                                      # all codes -8
    want = harness.unpack_int4(a).double() @ harness.unpack_int4(b).double().t()      # |C| <= 64 K: exact
    assert torch.equal(quest.matmul_int4_int4t_int32(a, b).double(), want)
