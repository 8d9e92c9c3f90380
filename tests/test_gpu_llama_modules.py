"""A packed model whose parts a user has replaced, hooked or run under another mode: the native calls stand in for modules only
where nothing is passed by."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = 'cuda:0'


def packed(seq=64, **options):
    from quest_amd import llama
    torch.manual_seed(21)
    cfg = llama.LlamaConfig(n_layer=2, n_embd=256, n_head=4, vocab_size=384, sequence_length=seq)
    model = llama.Llama(cfg).to(torch.bfloat16).to(DEV).eval()
    ids = torch.randint(0, cfg.vocab_size, (2, 40), generator=torch.Generator().manual_seed(22)).to(DEV)
    return llama.quantize_model(model, 'int4', **{'fuse_producers': True, **options}), ids


@pytest.mark.parametrize('fuse', [True, False])
@pytest.mark.parametrize('change', ['none', 'layernorm', 'identity', 'own_forward'])
def test_last_logits_are_the_modules_own(fuse, change):
    """The last position of all logits, which the modules themselves compute (bf16 outputs: 2^-8 of a logit each way, and a norm
    summed in another order)."""
    model, ids = packed(fuse_producers=fuse)
    if change == 'layernorm':
        model.transformer.ln_f = torch.nn.LayerNorm(256).to(DEV).bfloat16()
        model.transformer.ln_f.bias.data.fill_(0.5)
    elif change == 'identity':
        model.transformer.ln_f = torch.nn.Identity()
    elif change == 'own_forward':
        model.lm_head.forward = lambda x: torch.nn.functional.linear(x, model.lm_head.weight) + 3
    with torch.no_grad():
        last, every = model(ids)['logits'], model(ids, all_logits=True)['logits']
    want = every[:, -1:].double()
    assert (last.double() - want).norm() <= 2. ** -7 * want.norm()


@pytest.mark.parametrize('which', ['ln_f', 'lm_head', 'global'])
def test_hooks_on_the_norm_and_the_head_run(which):
    model, ids = packed()
    seen = []
    mods = {'ln_f': model.transformer.ln_f, 'lm_head': model.lm_head}
    if which == 'global':
        handle = torch.nn.modules.module.register_module_forward_hook(lambda m, *_: seen.append(m))
    else:
        handle = mods[which].register_forward_hook(lambda m, i, o: seen.append(m) or o * 2)
    try:
        with torch.no_grad():
            got = model(ids)['logits']
    finally:
        handle.remove()
    assert all(seen.count(mods[w]) == 1 for w in mods if which in (w, 'global'))
    if which == 'lm_head':                                   # what the hook returns is the output
        with torch.no_grad():
            want = 2 * model(ids)['logits'].double()
        assert (got.double() - want).norm() <= 2. ** -7 * want.norm()


def test_dense_model_is_traceable_under_no_grad():
    """No tensor of the forward leaves torch's view: a trace replayed on other ids follows them."""
    from quest_amd import llama
    torch.manual_seed(23)
    cfg = llama.LlamaConfig(n_layer=1, n_embd=128, n_head=2, vocab_size=64, sequence_length=16)
    model = llama.Llama(cfg).to(torch.bfloat16).to(DEV).eval().requires_grad_(False)
    a, b = (torch.randint(0, 64, (2, 9), generator=torch.Generator().manual_seed(s)).to(DEV) for s in (1, 2))
    with torch.no_grad():
        model(a)
        traced = torch.jit.trace(lambda ids: model(ids)['logits'], (a,), check_trace=False)
        assert torch.equal(traced(b), model(b)['logits'])


@pytest.mark.parametrize('batch,seq', [(1, 8), (2, 40), (4, 64)])
def test_a_hook_on_the_output_projection_is_the_blocks_output(batch, seq):
    """The projection is called, and what the hook returns is what the stream gets: with zeros, a block without attention."""
    model, _ = packed()
    ids = torch.randint(0, 384, (batch, seq), generator=torch.Generator().manual_seed(24)).to(DEV)
    calls = []
    for block in model.transformer.h:
        block.attn.c_proj.register_forward_hook(lambda m, i, o: calls.append(m) or torch.zeros_like(o))
    with torch.no_grad():
        got = model(ids, all_logits=True)['logits']
    assert len(calls) == 2
    for block in model.transformer.h:
        block.attn.c_proj._forward_hooks.clear()
        block.attn.c_proj.w_scale.zero_()
    with torch.no_grad():
        assert torch.equal(got, model(ids, all_logits=True)['logits'])


@pytest.mark.parametrize('part,method', [('attn', 'attention_core'), ('mlp', 'swiglu_quantized')])
def test_replaced_methods_of_a_fused_block_run(part, method):
    model, ids = packed()
    ids = ids[:1, :20]                                                 # few tokens: packed codes in front of the gated unit
    calls = []
    module = getattr(model.transformer.h[0], part)
    own = getattr(module, method)
    with torch.no_grad():
        want = model(ids)['logits']
        setattr(module, method, lambda *a, **k: calls.append(1) or own(*a, **k))
        assert torch.equal(model(ids)['logits'], want)
    assert calls


@pytest.mark.parametrize('seq', [8, 100])
def test_fused_block_under_autocast(seq):
    """Autocast to the model's own type keeps the logits; to the other one, the attention's output no longer has the type of the
    weights, which is refused."""
    model, _ = packed(seq=128)
    ids = torch.randint(0, 384, (1, seq), generator=torch.Generator().manual_seed(25)).to(DEV)
    with torch.no_grad():
        want = model(ids)['logits']
        with torch.autocast('cuda', dtype=torch.bfloat16):
            got = model(ids)['logits']                       # (its head is torch's then: one rounding apart)
            assert (got.double() - want.double()).norm() <= 2. ** -7 * want.double().norm()
        with torch.autocast('cuda', dtype=torch.float16), pytest.raises(AssertionError):
            model(ids)


@pytest.mark.parametrize('batch,seq', [(1, 8), (1, 40), (2, 100), (9, 512)])
@pytest.mark.parametrize('which', ['c_attn', 'c_proj', 'w12', 'down'])
def test_fused_block_with_scales_at_an_odd_element(batch, seq, which):
    """What one projection's kernels cannot read, others can: the same logits, and no half-updated stream."""
    from quest_amd import llama
    torch.manual_seed(27)
    cfg = llama.LlamaConfig(n_layer=2, n_embd=1024, n_head=8, vocab_size=64)
    model = llama.quantize_model(llama.Llama(cfg).to(torch.bfloat16).to(DEV).eval(), 'int4', fuse_producers=True)
    ids = torch.randint(0, 64, (batch, seq), generator=torch.Generator().manual_seed(28)).to(DEV)
    with torch.no_grad():
        want = model(ids)['logits']
        for block in model.transformer.h:
            w = {'c_attn': block.attn.c_attn, 'c_proj': block.attn.c_proj, 'w12': block.mlp.w12, 'down': block.mlp.c_proj}[which]
            w.w_scale = torch.cat([w.w_scale[:1], w.w_scale])[1:]
        assert torch.equal(model(ids)['logits'], want)
