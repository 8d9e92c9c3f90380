"""The work that users of this package have it do, as timed cases: W4A4 linear layers from one token to a long prefill,
the activation quantiser and the weight packer on their own, the layer as the separate steps of the `quest` call surface,
and whole forwards of the Llama models.  Every case is one call (or one short sequence of calls) of public entry points on
tensors and modules that a program holds; `draw` gives more cases of the same ranges.

Sizes: the 12-layer d = 1024 model and the 1600M model of `quest_amd.bench_e2e`, the layer shapes of
`quest_amd.bench_layer` (rows of 1024 to 11008, 1024 to 22016 channels) and 1 to 16384 tokens.
"""
import math

import torch

import quest_amd as quest
from quest_amd import harness, llama
from quest_amd.bench_e2e import MODELS

DTYPES = {'bf16': torch.bfloat16, 'fp16': torch.float16}
K_RANGE, N_RANGE, M_RANGE = (1024, 11008), (1024, 22016), (1, 16384)
LARGEST_LINEAR = (16384, 4096, 22016)                # (M, K, N): the most that a drawn layer may cost
MAX_MODEL_TOKENS = {'213m': 16384, '1600m': 1536}    # about the same work


def listed():
    return [
        # one token through an attention output projection: the smallest call, launch and host latency
        dict(name='linear decode 1', kind='linear', m=1, k=4096, n=4096, dtype='fp16', hadamard=True, bias=False),
        # a decoding batch through the MLP's down projection: the weights stream from HBM once
        dict(name='linear decode 13', kind='linear', m=13, k=11008, n=4096, dtype='bf16', hadamard=True, bias=False),
        # a short prompt through an up projection, with the module's default options (a bias, no transform)
        dict(name='linear 200 bias', kind='linear', m=200, k=4096, n=11008, dtype='bf16', hadamard=False, bias=True),
        # an eighth of the down projection's rows (tensor-parallel by 8: K = 11008 / 8 is no multiple of 128), ragged M
        dict(name='linear shard 333', kind='linear', m=333, k=1376, n=4096, dtype='fp16', hadamard=False, bias=False),
        # prefill through the up or gate projection: the headline size
        dict(name='linear prefill 4096', kind='linear', m=4096, k=4096, n=11008, dtype='fp16', hadamard=True, bias=False),
        # the longest prefill of the layer benchmark through its widest layer (gate and up together)
        dict(name='linear prefill 16384', kind='linear', m=16384, k=4096, n=22016, dtype='bf16', hadamard=True, bias=False),
        # the activation quantiser alone on heavy-tailed activations with outlier channels
        dict(name='quantize 8192', kind='quantize', m=8192, k=4096, dtype='bf16'),
        # packing a layer's weights when a model is loaded
        dict(name='pack weights', kind='pack', n=11008, k=4096, dtype='bf16', hadamard=True),
        # the layer as separate calls: transform, scale, codes, int32 product, scale epilogue; ragged M
        dict(name='steps 1000', kind='steps', m=1000, k=4096, n=4096, dtype='fp16'),
        # whole models, next-token logits of a batch of prompts: a short one, a large batch, a mid-sized ragged one
        dict(name='model 213m 1x37', kind='model', model='213m', batch=1, seq=37),
        dict(name='model 213m 32x512', kind='model', model='213m', batch=32, seq=512),
        dict(name='model 1600m 2x500', kind='model', model='1600m', batch=2, seq=500),
    ]


def _log_uniform(rng, low, high):
    return min(high, max(low, round(math.exp(rng.uniform(math.log(low), math.log(high))))))


def _whole(v, step, low):
    return max(low, v // step * step)


def draw(rng):
    """One more case: kinds in about the proportion of the list, sizes spread over the logarithm of their range."""
    kind = rng.choice(['linear'] * 6 + ['quantize', 'pack', 'steps', 'model', 'model', 'model'])
    dtype = rng.choice(sorted(DTYPES))
    if kind == 'model':
        model = rng.choice(sorted(MODELS))
        seq = _log_uniform(rng, 8, 512)
        batch = _log_uniform(rng, 1, max(1, min(64, MAX_MODEL_TOKENS[model] // seq)))
        return dict(kind=kind, model=model, batch=batch, seq=seq)
    hadamard = rng.random() < 0.6
    k = _log_uniform(rng, *K_RANGE)
    k = _whole(k, 128 if hadamard or kind != 'linear' else 32, K_RANGE[0])
    n = _log_uniform(rng, *N_RANGE)
    if rng.random() < 0.7:                            # most layers are whole 64s wide; any width is allowed
        n = _whole(n, 64, N_RANGE[0])
    if kind == 'pack':
        return dict(kind=kind, n=n, k=k, dtype=dtype, hadamard=hadamard)
    if kind == 'quantize':
        return dict(kind=kind, m=_log_uniform(rng, *M_RANGE), k=k, dtype=dtype)
    m_max = min(M_RANGE[1], LARGEST_LINEAR[0] * LARGEST_LINEAR[1] * LARGEST_LINEAR[2] // (k * n))
    if kind == 'steps':
        return dict(kind=kind, m=_log_uniform(rng, 1, min(4096, m_max)), k=k, n=n, dtype=dtype)
    return dict(kind=kind, m=_log_uniform(rng, 1, m_max), k=k, n=n, dtype=dtype, hadamard=hadamard,
                bias=rng.random() < 0.25)


def _activations(g, m, k, dtype, heavy_tails=False):
    """N(0, 1) rows; with heavy tails, Student-t with three degrees of freedom and one channel in a hundred 20 times up."""
    x = torch.randn(m, k, device='cuda', generator=g)
    if heavy_tails:
        chi2 = sum(torch.randn(m, k, device='cuda', generator=g).square_() for _ in range(3))
        x *= torch.rsqrt(chi2 / 3)
        x[:, torch.randperm(k, device='cuda', generator=g)[:max(1, k // 100)]] *= 20
    return x.to(dtype)


def _weight(g, n, k, dtype):
    return (torch.randn(n, k, device='cuda', generator=g) * 0.02).to(dtype)


@torch.inference_mode()
def prepare(case, seed):
    kind = case['kind']
    if kind == 'model':
        torch.manual_seed(seed)
        with torch.device('cuda'):
            net = llama.Llama(llama.LlamaConfig(**MODELS[case['model']])).to(torch.bfloat16).eval()
            ids = torch.randint(0, net.config.vocab_size, (case['batch'], case['seq']))
        return dict(kind=kind, net=llama.quantize_model(net, 'int4', fuse_producers=True), ids=ids)
    g = torch.Generator(device='cuda').manual_seed(seed)
    dtype = DTYPES[case['dtype']]
    if kind == 'quantize':
        return dict(kind=kind, x=_activations(g, case['m'], case['k'], dtype, heavy_tails=True))
    weight = _weight(g, case['n'], case['k'], dtype)
    if kind == 'pack':
        return dict(kind=kind, weight=weight, hadamard=case['hadamard'])
    x = _activations(g, case['m'], case['k'], dtype)
    if kind == 'linear':
        bias = _weight(g, 1, case['n'], dtype).view(-1) if case['bias'] else None
        return dict(kind=kind, x=x, layer=harness.Linear4bit.from_weight(weight, bias, use_hadamard=case['hadamard']))
    w_packed, w_scale, w_add, _ = harness.preprocess_weight(weight, use_hadamard=True)
    m, k, n = case['m'], case['k'], case['n']
    return dict(kind=kind, x=x, w_packed=w_packed, w_scale=w_scale, w_add=w_add,
                packed=torch.empty(m, k // 2, dtype=torch.uint8, device='cuda'),
                row_sum=torch.empty(m, 1, dtype=torch.int32, device='cuda'),
                product=torch.empty(m, n, dtype=torch.int32, device='cuda'))


@torch.inference_mode()
def run(state):
    kind = state['kind']
    if kind == 'linear':
        return state['layer'](state['x'])
    if kind == 'model':
        return state['net'](state['ids'])['logits']
    if kind == 'quantize':
        return quest.hadamard_quantize_int4(state['x'])
    if kind == 'pack':
        return harness.preprocess_weight(state['weight'], use_hadamard=state['hadamard'])
    x_had = quest.hadamard128(state['x'])
    scale = quest.find_scale_int4(x_had)
    quest.quantize_int4(x_had, scale, None, state['packed'], state['row_sum'])
    quest.matmul_int4_int4t_int32(state['packed'], state['w_packed'], state['product'])
    out = quest.add_mul_vv(state['row_sum'], scale, state['w_add'], state['w_scale'], state['product'])
    return x_had, scale, state['packed'], state['row_sum'], state['product'], out


def work(case):
    kind = case['kind']
    if kind == 'model':
        cfg = llama.LlamaConfig(**MODELS[case['model']])
        b, t, d = case['batch'], case['seq'], cfg.n_embd
        linear = cfg.linear_ops_per_token()
        # weights as nibbles, the embedding rows, the last positions' logits from the dense head; causal attention
        return dict(bytes=linear // 4 + b * t * (8 + 2 * d) + 2 * cfg.vocab_size * (d + b),
                    flops=linear * b * t + cfg.n_layer * 2 * b * t * t * d + 2 * b * d * cfg.vocab_size)
    k = case['k']
    if kind == 'pack':
        return dict(bytes=case['n'] * (2 * k + k // 2 + 2 + 4), flops=(7 if case['hadamard'] else 0) * case['n'] * k)
    m = case['m']
    if kind == 'quantize':
        return dict(bytes=m * (2 * k + k // 2 + 2 + 4), flops=7 * m * k)
    n = case['n']
    if kind == 'linear':
        return dict(bytes=2 * m * k + n * (k // 2 + 2 + (2 if case['bias'] else 0)) + 2 * m * n, flops=2 * m * n * k)
    # every call's inputs and outputs: transform, scale, codes, product, epilogue
    return dict(bytes=m * (4 * k + 2 * k + 2 * k + k // 2 + k // 2) + n * k // 2 + m * n * (4 + 4 + 2) + 12 * m + 6 * n,
                flops=2 * m * n * k)


def tolerance(case):
    # 16-bit float outputs.  Codes, sums and products of the quantiser follow its scale, which another order of the sum of
    # squares moves by one unit in the last place on about one row in ten thousand; a model's logits see such a step
    # through all of its 4-bit quantisers.
    if case['kind'] == 'model':
        return {'rel': 0.03}
    if case['kind'] in ('quantize', 'pack', 'steps'):
        return {'rel': 1e-2, 'max': 0.1, 'differ': 1e-3}
    return {'rel': 1e-2, 'max': 0.1}
