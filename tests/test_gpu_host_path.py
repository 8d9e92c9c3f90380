"""The native host path (csrc/host.cpp) against the Python statements it stands in for: the same bits, the same errors.
Declining every call makes the Python statements run."""
import sys
import threading
import time

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = 'cuda:0'


class _DeclinesAll:
    def __getattr__(self, _name):
        return lambda *_: None


@pytest.fixture
def python_path(monkeypatch):
    from quest_amd import api
    return lambda: monkeypatch.setattr(api, 'host', _DeclinesAll())


@pytest.mark.parametrize('dtype', [torch.bfloat16, torch.float16])
@pytest.mark.parametrize('lead,k,n,hadamard,bias', [((1,), 256, 64, True, False), ((3, 5), 384, 72, True, True), ((70,), 160, 33, False, True),
                                                    ((512,), 2048, 8448, True, False), ((512,), 2048, 8448, False, True)])
def test_linear_native_equals_python(python_path, dtype, lead, k, n, hadamard, bias):
    from quest_amd import harness
    g = torch.Generator(device=DEV).manual_seed(5)
    w = (torch.randn(n, k, device=DEV, generator=g) * 0.02).to(dtype)
    x = torch.randn(*lead, k, device=DEV, generator=g).to(dtype)
    layer = harness.Linear4bit.from_weight(w, torch.randn(n, device=DEV, generator=g).to(dtype) if bias else None, use_hadamard=hadamard)
    got = layer(x)
    strided = layer(x.repeat_interleave(2, -1)[..., ::2])          # not contiguous: the native path declines
    python_path()
    want = layer(x)
    assert got.shape == (*lead, n)
    assert torch.equal(got, want) and torch.equal(strided, want)


@pytest.mark.parametrize('batch,seq', [(1, 1), (1, 37), (3, 64), (2, 512)])
def test_block_native_equals_python(python_path, batch, seq):
    """Small, mid-sized and large-tile kernels, the packed and the tile form of the codes (hidden 2816, 256-wide tiles)."""
    from quest_amd import llama
    torch.manual_seed(3)
    with torch.device(DEV):
        net = llama.Llama(llama.LlamaConfig(n_layer=2, n_embd=2048, n_head=16, vocab_size=512)).to(torch.bfloat16).eval()
        ids = torch.randint(0, 512, (batch, seq))
    net = llama.quantize_model(net, 'int4', fuse_producers=True)
    with torch.no_grad():
        got = net(ids, all_logits=True)['logits']
        python_path()
        want = net(ids, all_logits=True)['logits']
    assert torch.equal(got, want)


@pytest.mark.parametrize('head_dim,seq,ours', [(64, 4096, True), (64, 4097, False), (64, 4200, False), (128, 2048, True), (128, 2049, False), (128, 4200, False)])
def test_sequences_beyond_the_pinned_bits_go_to_the_library(python_path, head_dim, seq, ours):
    """Where the attention kernel's bits are not the library's any more, a native block calls the library."""
    from quest_amd import llama
    torch.manual_seed(4)
    with torch.device(DEV):
        net = llama.Llama(llama.LlamaConfig(n_layer=1, n_embd=512, n_head=512 // head_dim, vocab_size=256, sequence_length=seq)).to(torch.bfloat16).eval()
        ids = torch.randint(0, 256, (1, seq))
    net = llama.quantize_model(net, 'int4', fuse_producers=True)
    with torch.no_grad():
        got, calls = _attention_calls(lambda: net(ids, all_logits=True)['logits'])
        assert calls == (0 if ours else 1)
        python_path()
        want = net(ids, all_logits=True)['logits']
    assert torch.equal(got, want)


@pytest.mark.parametrize('dtype', [torch.bfloat16, torch.float16])
@pytest.mark.parametrize('head_dim,backends,ours', [
    (64, None, True), (128, None, True), (32, None, False), (96, None, False), (64, ['EFFICIENT_ATTENTION'], False), (128, ['EFFICIENT_ATTENTION'], False),
    (64, ['EFFICIENT_ATTENTION', 'FLASH_ATTENTION'], False), (64, ['FLASH_ATTENTION', 'EFFICIENT_ATTENTION'], True), (64, ['FLASH_ATTENTION'], True)])
def test_attention_is_the_one_that_the_caller_chose(python_path, head_dim, backends, ours, dtype):
    """Heads that the attention kernel does not take, and any choice of backends in which flash is not the first, go to the library, with
    the bits of the Python statements.  (Never the math backend: its batched products on transposed operands have faulted.)"""
    import contextlib

    from torch.nn.attention import SDPBackend, sdpa_kernel

    from quest_amd import llama
    torch.manual_seed(5)
    with torch.device(DEV):
        net = llama.Llama(llama.LlamaConfig(n_layer=2, n_embd=384, n_head=384 // head_dim, vocab_size=256)).to(dtype).eval()
        ids = torch.randint(0, 256, (2, 100))
    net = llama.quantize_model(net, 'int4', fuse_producers=True)
    chosen = lambda: contextlib.nullcontext() if backends is None else sdpa_kernel([getattr(SDPBackend, b) for b in backends], set_priority=True)      # noqa: E731
    with torch.no_grad(), chosen():
        got, calls = _attention_calls(lambda: net(ids, all_logits=True)['logits'])
        assert calls == (0 if ours else 2)
        python_path()
        want = net(ids, all_logits=True)['logits']
    assert torch.equal(got, want)


def _attention_calls(call):
    """The call's result and how often it went to the library's attention."""
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CPU]) as prof:
        result = call()
    return result, sum(e.count for e in prof.key_averages() if e.key == 'aten::scaled_dot_product_attention')


def test_declined_calls_raise_as_before():
    import quest_amd as quest
    x = torch.zeros(4, 256, dtype=torch.bfloat16, device=DEV)
    with pytest.raises(AssertionError):
        quest.hadamard128(x, torch.empty(4, 128, dtype=torch.bfloat16, device=DEV))
    with pytest.raises(AssertionError):
        quest.find_scale_int4(x[:, ::2])
    with pytest.raises(RuntimeError):
        quest.find_scale_int4(torch.zeros(4, 12, dtype=torch.bfloat16, device=DEV))       # rows that are not whole eights
    with pytest.raises(RuntimeError):
        quest.quantize_int4(x, torch.ones(4, 1, dtype=torch.bfloat16, device='cpu'))


@pytest.mark.parametrize('native', [True, False])
@pytest.mark.parametrize('dtype,tokens,calls', [(torch.float16, 8, 2), (torch.float16, 48, 2), (torch.float16, 64, 2), (torch.float16, 65, 0),
                                                (torch.bfloat16, 200, 0)])
def test_few_fp16_tokens_take_torchs_silu(python_path, native, dtype, tokens, calls):
    """The kernels' gated unit rounds two of the fp16 gates another way than torch: up to 64 tokens it is torch's, in both
    statements of the block, which then agree to the bit."""
    from quest_amd import llama
    torch.manual_seed(6)
    with torch.device(DEV):
        net = llama.Llama(llama.LlamaConfig(n_layer=2, n_embd=1024, n_head=8, vocab_size=256)).to(dtype).eval()
        ids = torch.randint(0, 256, (1, tokens))
    net = llama.quantize_model(net, 'int4', fuse_producers=True)
    with torch.no_grad():
        want = net(ids, all_logits=True)['logits']
        if not native:
            python_path()
        with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CPU]) as prof:
            got = net(ids, all_logits=True)['logits']
    assert sum(e.count for e in prof.key_averages() if e.key == 'aten::silu') == calls
    assert torch.equal(got, want)


def test_an_option_without_a_truth_value_raises_its_own_error():
    import quest_amd as quest
    x = torch.randn(4, 256, device=DEV).bfloat16()
    before = x.clone()
    with pytest.raises(RuntimeError, match='Boolean value of Tensor'):
        quest.quantize_int4(x, torch.ones(4, 1, dtype=torch.bfloat16, device=DEV), do_dequantize=torch.ones(2))
    assert torch.equal(x, before)


@pytest.mark.parametrize('m,k,n', [(1, 4096, 512), (333, 1376, 4096), (2000, 1024, 512)])
def test_a_layer_chooses_its_kernels_in_native_code(monkeypatch, m, k, n):
    """A call that the host bounds is not kept waiting by the choice in Python (0.25 us of 12)."""
    from quest_amd import harness
    layer = harness.Linear4bit.from_weight((torch.randn(n, k, device=DEV) * .02).half())
    x = torch.randn(m, k, device=DEV).half()
    want = layer(x)

    def asked(*_):
        raise AssertionError('asked in Python')
    for name in ('prefers_e2m3', 'one_launch_on_tiles', 'tiles_k'):
        monkeypatch.setattr(harness, name, asked)
    assert torch.equal(layer(x), want)


@pytest.mark.parametrize('lines,fp6', [({}, True), ({'E2M3_MIN_K': 1664}, False), ({'E2M3_SHORT_ROWS_TOKENS': 5000, 'E2M3_MIN_K': 1664}, True), ({'MATRIX_PATH': 'int8'}, False)])
def test_the_native_choice_follows_the_module(monkeypatch, lines, fp6):
    from quest_amd import harness
    layer = harness.Linear4bit.from_weight((torch.randn(1536, 1536, device=DEV) * .02).bfloat16())
    x = torch.randn(4097, 1536, device=DEV).bfloat16()
    want = layer(x)
    for name, value in lines.items():
        monkeypatch.setattr(harness, name, value)
    assert harness.prefers_e2m3(4097, 1536, 1536) == fp6
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CUDA]) as prof:
        got = layer(x)
        torch.cuda.synchronize()
    assert any('e2m3' in e.key for e in prof.key_averages()) == fp6 and torch.equal(got, want)


@pytest.mark.parametrize('call', ['linear', 'block', 'last_logits', 'steps'])
def test_other_threads_run_during_native_calls(call):
    """The interpreter lock is free while a native call allocates and launches: with a switch interval that never ends, a thread
    that wants it gets it from there only."""
    import quest_amd as quest
    from quest_amd import harness, llama
    x = torch.randn(2, 1024, device=DEV).bfloat16()
    if call == 'linear':
        layer = harness.Linear4bit.from_weight(torch.randn(256, 1024, device=DEV).bfloat16())
        run = lambda: layer(x)                                                # noqa: E731
    elif call == 'steps':
        scale, packed = quest.find_scale_int4(x), torch.empty(2, 512, dtype=torch.uint8, device=DEV)
        run = lambda: (quest.hadamard128(x), quest.find_scale_int4(x), quest.quantize_int4(x, scale, x_int_packed=packed),      # noqa: E731
                       quest.matmul_int4_int4t_int32(packed, packed), quest.hadamard_quantize_int4(x))
    else:
        cfg = llama.LlamaConfig(n_layer=1, n_embd=1024, n_head=8, vocab_size=64)
        net = llama.quantize_model(llama.Llama(cfg).to(DEV).bfloat16().eval(), 'int4', fuse_producers=True)
        stream = torch.randn(2, 8, 1024, device=DEV).bfloat16()
        freqs = net.freqs_cis[:8].to(DEV)
        if call == 'block':
            run = lambda: net.transformer.h[0].forward_fused(stream, freqs)   # noqa: E731
        else:
            run = lambda: quest.api.host.last_logits(stream, None, net.transformer.ln_f.weight, 1e-5, net.lm_head.weight)   # noqa: E731
    with torch.no_grad():
        run()
        torch.cuda.synchronize()
        turns, stop, ready = [0], threading.Event(), threading.Event()

        def other():
            ready.set()
            while not stop.is_set():
                turns[0] += 1
                time.sleep(0)
        thread = threading.Thread(target=other)
        interval = sys.getswitchinterval()
        thread.start()
        ready.wait()
        try:
            sys.setswitchinterval(1000)
            before = turns[0]
            for _ in range(3000):
                run()
            after = turns[0]
        finally:
            stop.set()
            sys.setswitchinterval(interval)
            thread.join()
    assert after - before > 10


class _Recorder:
    """The native module with what it returns to whom."""

    def __init__(self, real):
        self.real, self.calls = real, []

    def __getattr__(self, name):
        def call(*a):
            self.calls.append((name, getattr(self.real, name)(*a)))
            return self.calls[-1][1]
        return call

    def took(self):
        return [name for name, result in self.calls if result is not None]


@pytest.fixture
def native(monkeypatch):
    from quest_amd import _lib, api
    recorder = _Recorder(_lib.host)
    monkeypatch.setattr(api, 'host', recorder)
    return recorder


def _calls(m, k, n, dtype, given):
    """Every function of the native module as a call of the package on fixed inputs: name -> function returning all outputs."""
    import quest_amd as quest
    from quest_amd import harness
    g = torch.Generator(device=DEV).manual_seed(m + k + n)
    x = torch.randn(m, k, device=DEV, generator=g).to(dtype)
    a, b = (torch.randint(0, 256, (r, k // 2), device=DEV, generator=g, dtype=torch.uint8) for r in (m, n))
    a_mul, b_mul = ((torch.rand(r, 1, device=DEV, generator=g) + 0.5).to(dtype) for r in (m, n))
    a_add, b_add = (torch.randint(-99, 99, (r, 1), device=DEV, generator=g, dtype=torch.int32) for r in (m, n))
    c = torch.randint(-9999, 9999, (m, n), device=DEV, generator=g, dtype=torch.int32)
    out = lambda *shape, t=dtype: torch.empty(*shape, dtype=t, device=DEV) if given else None      # noqa: E731

    def quantize():
        y, outs = x.clone(), (torch.empty(m, k, dtype=torch.int8, device=DEV), torch.empty(m, k // 2, dtype=torch.uint8, device=DEV),
                              torch.empty(m, 1, dtype=torch.int32, device=DEV))
        return quest.quantize_int4(y, a_mul, *(outs if given else (None, outs[1], None)), do_dequantize=given)
    return dict(
        gemm=lambda: quest.fused_matmul_dequantize_int4_int4t_bf16(a, b, a_add, b_add, a_mul, b_mul, out(m, n)),
        matmul_int32=lambda: quest.matmul_int4_int4t_int32(a, b, out(m, n, t=torch.int32)),
        find_scale=lambda: quest.find_scale_int4(x, out(m, 1)),
        quantize=quantize,
        add_mul_vv=lambda: quest.add_mul_vv(a_add, a_mul, b_add, b_mul, c, out(m, n)),
        hadamard128=lambda: quest.hadamard128(x, out(m, k), 2. ** -3.5),
        hadamard_quantize=lambda: quest.hadamard_quantize_int4(x, out(m, 1), out(m, k // 2, t=torch.uint8), out(m, 1, t=torch.int32), scale_rule='absmax'),
        pack_weight=lambda: harness.preprocess_weight(x, use_hadamard=given, w_scale_mode='absmax' if given else 'rms')[:3],
        linear=lambda: harness.linear_forward(x, b, b_mul, b_add, use_hadamard=given, out=out(m, n)))


NAMES = ['gemm', 'matmul_int32', 'find_scale', 'quantize', 'add_mul_vv', 'hadamard128', 'hadamard_quantize', 'pack_weight', 'linear']


@pytest.mark.parametrize('dtype', [torch.bfloat16, torch.float16])
@pytest.mark.parametrize('given', [False, True])
@pytest.mark.parametrize('m,k,n', [(37, 256, 72), (1, 384, 33), (333, 1152, 1001)])
@pytest.mark.parametrize('name', NAMES)
def test_every_call_goes_native_and_equals_python(native, monkeypatch, name, m, k, n, given, dtype):
    from quest_amd import api
    call = _calls(m, k, n, dtype, given)[name]
    got = call()
    assert native.took() == [name]
    monkeypatch.setattr(api, 'host', _DeclinesAll())
    want = call()
    for x, y in zip(*((r if isinstance(r, tuple) else (r,)) for r in (got, want))):
        assert (x is None and y is None) or (torch.equal(x, y) and x.shape == y.shape and x.dtype == y.dtype)


def test_which_layers_and_blocks_go_native(native):
    """Plain ones do, down to the last logits; a strided input and a bias of another type do not."""
    from quest_amd import harness, llama
    layer = harness.Linear4bit.from_weight(torch.randn(72, 256, device=DEV).bfloat16(), torch.zeros(72, device=DEV).bfloat16())
    x = torch.randn(3, 512, device=DEV).bfloat16()
    native.calls.clear()
    layer(x[:, :256].contiguous())
    assert native.took() == ['linear']
    native.calls.clear()
    layer(x[:, ::2])
    assert [c for c in native.calls if c[0] == 'linear'][0][1] is None
    native.calls.clear()
    layer.bias = torch.nn.Parameter(layer.bias.float(), requires_grad=False)
    layer(x[:, :256].contiguous())
    assert [c for c in native.calls if c[0] == 'linear'][0][1] is None
    net = llama.quantize_model(llama.Llama(llama.LlamaConfig(n_layer=3, n_embd=1024, n_head=8, vocab_size=64)).to(DEV).bfloat16().eval(), 'int4',
                               fuse_producers=True)
    for batch, seq in ((1, 1), (2, 37), (3, 100), (9, 500)):
        native.calls.clear()
        with torch.no_grad():
            net(torch.randint(0, 64, (batch, seq), device=DEV))
        assert native.took() == ['block'] * 3 + ['last_logits']
