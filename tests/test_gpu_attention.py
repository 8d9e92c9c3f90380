"""The causal attention kernel: the bits of torch's own kernel over the lengths where its steps, blocks and tiles begin and end, its
error against fp64, and what lies beyond a sequence's last row."""
import math

import pytest
import torch
from torch.nn import functional as F

from quest_amd import _lib

pytestmark = pytest.mark.gpu
LENGTHS = [1, 2, 15, 16, 17, 31, 32, 33, 63, 64, 65, 95, 96, 127, 128, 129, 160, 191, 192, 255, 256, 257, 300, 383, 384, 385, 447, 500,
           511, 512, 513, 700, 1000, 1024, 2048, 2049, 3000, 4095, 4096]

SAME_BITS = {64: 4096, 128: 2048}                            # QUEST_ATTENTION_SAME_BITS: longest sequences with the library's bits


def attend(qkv, heads, out=None):
    b, t, c3 = qkv.shape
    out = torch.empty(b, t, c3 // 3, dtype=qkv.dtype, device='cuda') if out is None else out
    _lib.check(_lib.load().quest_causal_attention(_lib.ptr(out), _lib.ptr(qkv), b, t, heads, c3 // 3 // heads, _lib.DTYPE_CODE[qkv.dtype],
                                                  _lib.stream_of(qkv)), 'quest_causal_attention')
    return out


def parts(qkv, heads):
    b, t, c3 = qkv.shape
    return [z.view(b, t, heads, -1).transpose(1, 2) for z in qkv.split(c3 // 3, dim=2)]


def inputs(b, t, heads, d, dtype, amplitude, seed):
    g = torch.Generator(device='cuda').manual_seed(seed)
    return (torch.randn(b, t, 3 * heads * d, device='cuda', generator=g) * amplitude).to(dtype)


@pytest.mark.parametrize('dtype', [torch.bfloat16, torch.float16])
@pytest.mark.parametrize('t,d', [(t, d) for t in LENGTHS for d in SAME_BITS if t <= SAME_BITS[d]])
def test_bits_of_the_library_kernel(t, d, dtype):
    heads = 5
    for b, amplitude in ((1, 1.0), (3, 4.0)):
        qkv = inputs(b, t, heads, d, dtype, amplitude, 10 * t + b)
        q, k, v = parts(qkv, heads)
        want = F.scaled_dot_product_attention(q, k, v, is_causal=True).transpose(1, 2).reshape(b, t, -1)
        assert torch.equal(attend(qkv, heads), want)


@pytest.mark.parametrize('dtype', [torch.bfloat16, torch.float16])
@pytest.mark.parametrize('t,d', [(1, 64), (29, 128), (64, 64), (200, 64), (333, 128), (512, 64)])
def test_error_against_fp64(t, d, dtype):
    """An output is a sum of probabilities p_i <= 1, each rounded to dtype, times v_i, divided by the unrounded sum l of the p_i, and
    rounded once more: |error| <= u (sum p_i |v_i| / l + |out|), u = half a unit in the last place, plus fp32 noise (a tenth of
    it is allowed for: some hundred operations at 2^-24)."""
    heads = 3
    qkv = inputs(2, t, heads, d, dtype, 1.0, t)
    q, k, v = (z.double().cpu() for z in parts(qkv, heads))
    s = (q @ k.transpose(-1, -2)) / math.sqrt(d)
    p = s.masked_fill(torch.ones(t, t, dtype=torch.bool).triu(1), float('-inf')).softmax(-1)
    want, spread = p @ v, p @ v.abs()
    got = attend(qkv, heads).view(2, t, heads, d).transpose(1, 2).double().cpu()
    u = 2.0 ** (-8 if dtype == torch.bfloat16 else -11)
    assert ((got - want).abs() <= 1.1 * u * (spread + want.abs()) + 1e-7).all()      # (fp16's subnormal probabilities: 2^-25 each)


@pytest.mark.parametrize('t', [5, 40, 200, 300])
@pytest.mark.parametrize('d', [64, 128])
def test_nothing_crosses_a_sequence_end(t, d):
    heads = 2
    qkv = inputs(3, t, heads, d, torch.bfloat16, 1.0, t)
    want = attend(qkv, heads)
    qkv[1] = float('nan')                                    # the rows before and after a sequence's own
    out = torch.full((t * 3 + 256, heads * d), 7.0, dtype=torch.bfloat16, device='cuda')
    attend(qkv, heads, out)
    assert torch.equal(out[:t], want[0]) and torch.equal(out[2 * t:3 * t], want[2])
    assert out[t:2 * t].isnan().all() and (out[3 * t:] == 7).all()


@pytest.mark.parametrize('dtype', [torch.bfloat16, torch.float16])
@pytest.mark.parametrize('d', [64, 128])
@pytest.mark.parametrize('t', [1, 5, 16, 30, 64, 127, 200, 300, 500])
def test_scores_of_minus_infinity_add_nothing(t, d, dtype):
    """The first half of the keys score -inf for every query: whole steps, and whole rows, of nothing else.  The rows behind them are
    those of the other keys, whichever order they are summed in; the first ones are zero, as the library's are."""
    qkv = inputs(1, t, 1, d, dtype, 1.0, t)
    half = (t + 1) // 2
    qkv[0, :, 0] = qkv[0, :, 0].abs() + 0.1
    qkv[0, :half, d:2 * d] = 0
    qkv[0, :half, d] = float('-inf')
    q, k, v = parts(qkv, 1)
    want = F.scaled_dot_product_attention(q, k, v, is_causal=True).transpose(1, 2).reshape(1, t, d)
    got = attend(qkv, 1)
    assert torch.equal(got, want) and not got[0, :half].any() and got.isfinite().all()


def test_refused_calls():
    lib, qkv = _lib.load(), torch.zeros(1, 8, 3 * 96, dtype=torch.bfloat16, device='cuda')
    out = torch.zeros(1, 8, 96, dtype=torch.bfloat16, device='cuda')
    call = lambda o, x, *sizes: lib.quest_causal_attention(o, x, *sizes, 0, _lib.stream_of(qkv))
    assert call(out.data_ptr(), qkv.data_ptr(), 1, 8, 1, 96) != 0 and call(out.data_ptr(), qkv.data_ptr(), 1, 8, 3, 32) != 0
    assert call(out.data_ptr(), qkv.data_ptr() + 2, 1, 2, 1, 64) != 0 and call(None, qkv.data_ptr(), 1, 2, 1, 64) != 0
    assert call(out.data_ptr(), qkv.data_ptr(), 1, 0, 1, 64) != 0 and call(out.data_ptr(), qkv.data_ptr(), 1, 1 << 30, 1, 64) != 0
    torch.cuda.synchronize()
    assert not out.any()


@pytest.mark.parametrize('name', ['213m', '1600m'])
def test_both_twins_of_the_sweep_run_the_same_attention(name):
    """Fused blocks minus the same with no-op GEMMs prices the GEMMs: neither may run the library's attention."""
    from quest_amd import bench_e2e, llama
    cfg = llama.LlamaConfig(**{**bench_e2e.MODELS[name], 'n_layer': 1, 'vocab_size': 256})
    ids = torch.randint(0, 256, (2, 70), device='cuda')
    for mode in ('fused', 'fused_noop'):
        net = bench_e2e.build(mode, cfg, torch.device('cuda'))
        with torch.inference_mode(), torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CPU]) as prof:
            assert net.hidden_states(ids).isfinite().all()
        assert not [e.key for e in prof.key_averages() if 'scaled_dot_product' in e.key]
