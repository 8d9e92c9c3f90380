"""The operand forms derived from packed weights (E2M3 tiles, interleaved gate / up rows): made when the buffers get their content,
never by a forward call, and never used for other content."""
import copy
import io

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = 'cuda:0'
M, K, N = 96, 2048, 1024                      # a size the FP6 kernels take


@pytest.fixture
def harness():
    from quest_amd import harness as h
    assert h.prefers_e2m3(M, K, N)
    return h


def weight(seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    return (torch.randn(N, K, device=DEV, generator=g) * 0.02).bfloat16()


def rows(m=M):
    return torch.randn(m, K, device=DEV, generator=torch.Generator(device=DEV).manual_seed(9)).bfloat16()


def on_int8(harness, layer, x):
    return harness.linear_forward(x, layer.w_int_packed, layer.w_scale, layer.w_add, use_hadamard=layer.use_hadamard)


def model(seed, inference=False):
    from quest_amd import llama
    torch.manual_seed(seed)
    cfg = llama.LlamaConfig(n_layer=2, n_embd=1024, n_head=8, vocab_size=256, sequence_length=128)
    with torch.inference_mode(inference):
        return llama.quantize_model(llama.Llama(cfg).to(DEV).bfloat16().eval(), 'int4', fuse_producers=True)


IDS = torch.randint(0, 256, (2, 100), generator=torch.Generator().manual_seed(8))


@torch.inference_mode()
def logits(net):
    return net(IDS.to(DEV), all_logits=True)['logits']


@pytest.mark.parametrize('how', ['packed', 'packed in inference mode', 'loaded', 'loaded in inference mode', 'assigned', 'moved', 'deep copy', 'pickled'])
def test_no_forward_converts_weights(harness, monkeypatch, how):
    """Whatever gave the layer its content, its tiles are there before the first call."""
    with torch.inference_mode('inference' in how):
        layer = harness.Linear4bit.from_weight(weight(1), use_hadamard=True)
        if how in ('loaded', 'loaded in inference mode', 'assigned'):
            other = layer
            layer = harness.Linear4bit.empty(K, N, device=DEV, dtype=torch.bfloat16, use_hadamard=True)
            layer.load_state_dict(other.state_dict(), assign=how == 'assigned')
    if how == 'moved':
        layer = layer.to('cpu').to(DEV)
    elif how == 'deep copy':
        layer = copy.deepcopy(layer)
    elif how == 'pickled':
        file = io.BytesIO()
        torch.save(layer, file)
        file.seek(0)
        layer = torch.load(file, weights_only=False)
    want = on_int8(harness, layer, rows())

    def convert(_):
        raise AssertionError('a forward call converted weights')
    monkeypatch.setattr(harness, 'weight_tiles', convert)
    assert layer.tiles_for(M) is not None
    assert torch.equal(layer(rows()), want)


@pytest.mark.parametrize('inference', [False, True])
def test_writes_into_the_buffer_show(harness, inference):
    """A reload or a write by hand under inference mode reaches calls of every size; by hand, the packed codes serve until the tiles
    are laid out again."""
    with torch.inference_mode(inference):
        layer, other, third = (harness.Linear4bit.from_weight(weight(s), use_hadamard=True) for s in (1, 2, 3))
        layer(rows())
        layer.load_state_dict(other.state_dict())
        assert layer.tiles_for(M) is not None
        assert torch.equal(layer(rows()), on_int8(harness, other, rows()))
        for name in ('w_int_packed', 'w_scale', 'w_add'):
            getattr(layer, name).copy_(getattr(third, name))
        want = on_int8(harness, third, rows())
        assert layer.tiles_for(M) is None and torch.equal(layer(rows()), want)
        a_scale, a_tiles = harness.quest.hadamard_quantize_e2m3(rows())
        assert torch.equal(layer.forward_tiles(a_scale, a_tiles), want)
        layer.lay_out_tiles()
        assert layer.tiles_for(M) is not None and torch.equal(layer(rows()), want)


@pytest.mark.parametrize('native', [True, False])
@pytest.mark.parametrize('entry', ['quantize_int4', 'hadamard_quantize_int4', 'hadamard_quantize_e2m3'])
def test_quantisers_write_into_the_buffers(harness, monkeypatch, entry, native):
    """Weights packed straight into a layer's buffers by the quantisers, whose writes torch does not see by itself."""
    api = harness.quest
    layer, fresh = harness.Linear4bit.from_weight(weight(6), use_hadamard=False), weight(7)
    want = on_int8(harness, harness.Linear4bit.from_weight(fresh, use_hadamard=False), rows())
    if not native:
        class Declines:
            def __getattr__(self, _name):
                return lambda *_: None
        monkeypatch.setattr(api, 'host', Declines())
    sums = torch.empty(N, 1, dtype=torch.int32, device=DEV)
    before = layer.w_scale._version
    if entry == 'quantize_int4':
        api.find_scale_int4(fresh, layer.w_scale)
        api.quantize_int4(fresh, layer.w_scale, x_int_packed=layer.w_int_packed, x_int_row_sum=sums)
    elif entry == 'hadamard_quantize_int4':
        api.hadamard_quantize_int4(fresh, layer.w_scale, layer.w_int_packed, sums, hadamard_scale=0.)
    else:
        api.hadamard_quantize_e2m3(fresh, layer.w_scale, None, layer.w_int_packed, sums, hadamard_scale=0.)
    layer.w_add.copy_(sums + K // 2)
    assert layer.w_scale._version > before
    assert torch.equal(layer(rows()), want)
    layer.lay_out_tiles()
    assert layer.tiles_for(M) is not None and torch.equal(layer(rows()), want)


def test_first_call_inside_a_capture(harness):
    """Warmed with one token only, captured at many, and called eagerly before and between the replays."""
    layer, x = harness.Linear4bit.from_weight(weight(4), use_hadamard=True), rows()
    want = on_int8(harness, layer, x)
    layer(x[:1])
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = layer(x)
    for _ in range(3):
        assert torch.equal(layer(x), want)
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want)


@pytest.mark.parametrize('inference', [False, True])
def test_captured_calls_follow_a_reload(harness, inference):
    """load_state_dict writes the packed codes in place, and so their other forms: a graph captured before it runs the new weights, for a
    layer and for a fused model (whose gate / up rows are a copy of their own)."""
    with torch.inference_mode(inference):
        layer, other = (harness.Linear4bit.from_weight(weight(s), use_hadamard=True) for s in (1, 2))
    nets, x, ids = (model(1, inference), model(2, inference)), rows(), IDS.to(DEV)
    calls = ((layer, other, lambda m: m(x)), (*nets, lambda m: m(ids, all_logits=True)['logits']))
    for kept, new, call in calls:
        with torch.no_grad():
            want = call(new).clone()
            side = torch.cuda.Stream()
            side.wait_stream(torch.cuda.current_stream())
            with torch.cuda.stream(side):
                call(kept)
            torch.cuda.current_stream().wait_stream(side)
            graph = torch.cuda.CUDAGraph()
            with torch.cuda.graph(graph):
                out = call(kept)
            for _ in range(2):                                         # (the second load writes what the first one left in place)
                with torch.inference_mode(inference):
                    kept.load_state_dict(new.state_dict())
                filler = [torch.full((1 << 20,), 0x55, dtype=torch.uint8, device=DEV) for _ in range(32)]      # takes up freed memory
                graph.replay()
                torch.cuda.synchronize()
                assert torch.equal(out, want) and torch.equal(call(kept), want)
                del filler


def test_a_move_to_where_it_is_keeps_one_copy(harness):
    net = model(1)
    net.to(DEV)
    assert all(b.mlp.w12._tiles is None and b.mlp.glu_tiles is not None and b.mlp.kept_glu() is not None for b in net.transformer.h)


def test_packing_a_fused_model_lays_out_what_it_keeps(harness, monkeypatch):
    made, convert = [], harness.weight_tiles
    monkeypatch.setattr(harness, 'weight_tiles', lambda *a: made.append(convert(*a)) or made[-1])
    net = model(1)
    kept = [t for b in net.transformer.h for t in (b.attn.c_attn._kept_tiles(), b.attn.c_proj._kept_tiles(), b.mlp.glu_tiles, b.mlp.c_proj._kept_tiles())]
    assert len(made) == len(kept) and {t.data_ptr() for t in made} == {t.data_ptr() for t in kept}


def test_first_calls_on_two_streams(harness):
    """Both streams wait for the packing stream only."""
    layer, x = harness.Linear4bit.from_weight(weight(5), use_hadamard=True), rows()
    want = on_int8(harness, layer, x)
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    outs = []
    for s in streams:
        s.wait_stream(torch.cuda.current_stream())
    for s in streams:
        with torch.cuda.stream(s):
            outs.append(layer(x))
    torch.cuda.synchronize()
    assert all(torch.equal(o, want) for o in outs)


@pytest.mark.parametrize('inference', [False, True])
@pytest.mark.parametrize('how', ['loaded', 'written', 'moved', 'deep copy'])
def test_fused_model_follows_its_buffers(monkeypatch, how, inference):
    from quest_amd import harness
    net, other = model(1, inference), model(2, inference)
    want, own = logits(other), logits(net)
    assert not torch.equal(own, want)
    if how == 'loaded':
        with torch.inference_mode(inference):
            net.load_state_dict(other.state_dict())
    elif how == 'written':
        with torch.inference_mode(inference):
            for name, t in net.state_dict().items():
                t.copy_(other.state_dict()[name])
    elif how == 'moved':
        with torch.inference_mode(inference):
            net, want = net.to('cpu').to(DEV), own
    else:
        net, want = copy.deepcopy(net), own
    if how != 'written':
        def convert(_):
            raise AssertionError('a forward call converted weights')
        monkeypatch.setattr(harness, 'weight_tiles', convert)
    assert torch.equal(logits(net), want)
