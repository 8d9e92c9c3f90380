"""The FP6 layer in one launch against the activation kernel and the GEMM one after the other: both forms of the workgroup (rows of 5 to 8 and of 9 to
16 blocks), one channel tile at a time and two, the edges of token and channel tiles, more tiles than workgroups, the norm in front, every epilogue, degenerate rows."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = 'cuda:0'
PLAIN, SWIGLU, ADD, ROPE, BIAS = range(5)
SIZES = [(37, 1024, 3072), (1, 640, 32), (32, 1024, 1024), (33, 1152, 40), (12, 2048, 5632), (128, 2048, 1000), (5, 768, 4100), (13, 896, 22016), (256, 1024, 8),
         (31, 1920, 4096), (65, 1664, 264), (8, 1280, 22000), (128, 1024, 8136), (37, 1024, 22016), (70, 768, 5670)]
RAGGED = [(9, 1376, 4096), (40, 672, 300), (64, 2016, 96), (17, 544, 5000)]                     # whole 32s, without norm and transform
REFUSED = [(257, 1024, 512), (8, 512, 512), (8, 2176, 512), (160, 1024, 8192), (64, 2048, 6144)]


def _call(l):
    from quest_amd import _lib
    return _lib.load().quest_linear_e2m3_fused(ctypes.byref(l), torch.cuda.current_stream().cuda_stream)


def _operands(m, k, n, dtype):
    from quest_amd import harness
    g = torch.Generator(device=DEV).manual_seed(m * k + n)
    x = torch.randn(m, k, device=DEV, generator=g).to(dtype)
    if m > 3:
        x[1], x[2, 5], x[3, 7] = 0, float('nan'), float('inf')
    w = torch.randint(0, 256, (n, k // 2), dtype=torch.uint8, device=DEV, generator=g)
    from quest_amd.api import int4_to_e2m3_tiles_padded as padded
    return dict(x=x, tiles=harness.weight_tiles(w) if k % 128 == 0 else padded(w), scale=(torch.rand(n, 1, device=DEV, generator=g) * .1).to(dtype), norm=torch.rand(k, device=DEV, generator=g).to(dtype),
                bias=torch.randn(n, device=DEV, generator=g).to(dtype), before=torch.randn(m, n, device=DEV, generator=g).to(dtype))


def _arguments(o, out, m, k, n, had_scale, norm, epilogue, rope=(None, 0, 0, 0)):
    from quest_amd import _lib
    l = _lib.FusedLinear()
    l.out, l.x, l.norm_weight, l.eps = out.data_ptr(), o['x'].data_ptr(), o['norm'].data_ptr() if norm else 0, 1e-5
    l.w_tiles, l.w_scale, l.epilogue, l.bias = o['tiles'].data_ptr(), o['scale'].data_ptr(), epilogue, o['bias'].data_ptr()
    l.freqs_cis, l.seq_len, l.rot_cols, l.head_dim = 0 if rope[0] is None else rope[0].data_ptr(), *rope[1:]
    l.size_m, l.size_k, l.size_n, l.had_scale, l.dtype = m, k, n, had_scale, _lib.DTYPE_CODE[out.dtype]
    return l


def _two_launches(o, m, k, n, had_scale, norm, epilogue, rope, out):
    """The same through the separate entry points: quantiser, then the GEMM with the epilogue."""
    from quest_amd import _lib
    lib, st, code = _lib.load(), torch.cuda.current_stream().cuda_stream, _lib.DTYPE_CODE[out.dtype]
    a_scale, a = torch.empty(m, dtype=out.dtype, device=DEV), torch.empty(lib.quest_e2m3_tiles_bytes(m, k), dtype=torch.uint8, device=DEV)
    kt = (k + 127) // 128 * 128
    if kt != k:
        a = torch.empty(lib.quest_e2m3_tiles_bytes(m, kt), dtype=torch.uint8, device=DEV)
        rc = lib.quest_quantize_e2m3_padded(o['x'].data_ptr(), a_scale.data_ptr(), a.data_ptr(), k, m, code, st)
    elif norm:
        rc = lib.quest_rmsnorm_hadamard_quantize_e2m3(o['x'].data_ptr(), o['norm'].data_ptr(), 1e-5, a_scale.data_ptr(), a.data_ptr(), 0, k, m, had_scale, code, st)
    else:
        rc = lib.quest_hadamard_quantize_e2m3(o['x'].data_ptr(), a_scale.data_ptr(), a.data_ptr(), 0, 0, 0, k, m, had_scale, code, st)
    assert rc == 0
    k = kt
    p = [out.data_ptr(), a.data_ptr(), o['tiles'].data_ptr(), a_scale.data_ptr(), o['scale'].data_ptr()]
    if epilogue == ROPE:
        rc = lib.quest_fused_matmul_dequantize_e2m3(*p, m, k, n, code, st) or lib.quest_rope_interleaved(out.data_ptr(), rope[0].data_ptr(), m, rope[1], n, rope[2], rope[3], code, st)
    elif epilogue == BIAS:
        rc = lib.quest_fused_matmul_dequantize_bias_e2m3(*p, o['bias'].data_ptr(), m, k, n, code, st)
    else:
        name = {PLAIN: '', SWIGLU: 'swiglu_', ADD: 'add_'}[epilogue]
        rc = getattr(lib, f'quest_fused_matmul_dequantize_{name}e2m3')(*p, m, k, n, code, st)
    assert rc == 0
    return out


@pytest.mark.parametrize('dtype', [torch.bfloat16, torch.float16])
@pytest.mark.parametrize('m,k,n', SIZES + RAGGED)
def test_equals_the_two_launches(dtype, m, k, n):
    from quest_amd import harness
    o = _operands(m, k, n, dtype)
    for norm, had_scale, epilogue in [(a, b, e) for a in (False, True) for b in (harness.HADAMARD_ENTRY, 0.) for e in (PLAIN, SWIGLU, ADD, ROPE, BIAS)
                                      if k % 128 == 0 or not (a or b)]:
        rope, width = (None, 0, 0, 0), n
        if epilogue == SWIGLU and n % 8 == 0:
            width = n // 2
        elif epilogue == SWIGLU:
            continue
        if epilogue == ROPE:
            if n < 96 or n % 8:
                continue
            seq, half = 19, 16                     # short and odd sequences; a quarter of the channels is not turned
            rope = (torch.randn(seq, half, 2, device=DEV), seq, n // 4 * 3 // 32 * 32, 2 * half)
        start = o['before'] if epilogue == ADD else torch.full((m, width), 7., dtype=dtype, device=DEV)
        guarded = torch.cat([start, torch.full((1, width), 7., dtype=dtype, device=DEV)])
        want = _two_launches(o, m, k, n, had_scale, norm, epilogue, rope, start.clone())
        assert _call(_arguments(o, guarded, m, k, n, had_scale, norm, epilogue, rope)) == 0
        same = (guarded[:m] == want) | (guarded[:m].isnan() & want.isnan())
        assert bool(same.all()), (norm, had_scale, epilogue, int((~same).sum()))
        assert bool((guarded[m] == 7.).all())


@pytest.mark.parametrize('m,k,n', REFUSED)
def test_other_sizes_are_refused(m, k, n):
    from quest_amd import harness
    o = _operands(m, k, n, torch.bfloat16)
    out = torch.full((m, n), 7., dtype=torch.bfloat16, device=DEV)
    assert _call(_arguments(o, out, m, k, n, harness.HADAMARD_ENTRY, False, PLAIN)) != 0 and bool((out == 7.).all())


def test_a_refusal_costs_the_host_little():
    """Two launches follow it, in calls that the host bounds: no question to the runtime (0.3 us) before the sizes have been looked at."""
    import time
    from quest_amd import _lib, harness
    call, stream = _lib.load().quest_linear_e2m3_fused, torch.cuda.current_stream().cuda_stream

    def best(m, k, n):
        o = _operands(m, k, n, torch.bfloat16)
        l = _arguments(o, torch.empty(m, n, dtype=torch.bfloat16, device=DEV), m, k, n, harness.HADAMARD_ENTRY, False, PLAIN)
        refer, times = ctypes.byref(l), []
        for _ in range(200):
            start = time.perf_counter()
            for _ in range(100):
                call(refer, stream)
            times.append(time.perf_counter() - start)
        return min(times)
    assert best(160, 1024, 8192) < 1.7 * best(257, 1024, 512)            # 1.2; 2.2 with the question


@pytest.mark.parametrize('m,k,n,hadamard,bias', [(9, 1024, 3072, True, False), (16, 2048, 8192, False, True), (37, 1376, 1000, False, True), (64, 1024, 5600, True, True),
                                                 (64, 1920, 2052, True, False), (30, 640, 12000, False, False), (48, 1536, 9, True, False), (128, 1024, 6400, True, True)])
def test_layer_equals_the_int8_path(monkeypatch, m, k, n, hadamard, bias):
    from quest_amd import harness
    g = torch.Generator(device=DEV).manual_seed(m + k + n)
    weight, x = (torch.randn(n, k, device=DEV, generator=g) * 0.02).bfloat16(), torch.randn(m, k, device=DEV, generator=g).bfloat16()
    layer = harness.Linear4bit.from_weight(weight, torch.randn(n, device=DEV, generator=g).bfloat16() if bias else None, use_hadamard=hadamard)
    assert harness.prefers_e2m3(m, harness.tiles_k(k, hadamard), n)
    with torch.no_grad():
        got = layer(x)
        monkeypatch.setattr(harness, 'MATRIX_PATH', 'int8')
        assert torch.equal(got, layer(x))


@pytest.mark.parametrize('dtype', [torch.bfloat16, torch.float16])
@pytest.mark.parametrize('batch,seq', [(1, 1), (1, 5), (3, 7), (1, 32), (2, 37)])
def test_model_equals_the_int8_path(monkeypatch, dtype, batch, seq):
    from quest_amd import harness, llama
    torch.manual_seed(batch + seq)
    with torch.device(DEV):
        net = llama.Llama(llama.LlamaConfig(n_embd=1024, n_layer=2, n_head=16, vocab_size=512, sequence_length=64)).to(dtype).eval()
        ids = torch.randint(0, 512, (batch, seq))
    net = llama.quantize_model(net, 'int4', fuse_producers=True)
    with torch.inference_mode():
        got = net(ids)['logits']
        monkeypatch.setattr(harness, 'MATRIX_PATH', 'int8')
        assert torch.equal(got, net(ids)['logits'])
