"""Decode graph sizes between the listed ones: which are added, and that a step in one of them gives what the
same step gives without graphs."""
import pytest
import torch

from mlopamd.models import build_model
from mlopamd.models.config import get_config
from mlopamd.runtime.engine import Engine, EngineConfig, fill_buckets

LISTED = EngineConfig.graph_buckets


@pytest.mark.parametrize("listed, want", [
    ((1, 2, 4, 8, 16, 32), [1, 2, 4, 8, 16, 32]),
    ((32, 64, 128), [32, 48, 64, 80, 96, 112, 128]),
    ((128, 256), [128, 160, 192, 224, 256]),
    ((256, 512), [256, 320, 384, 448, 512]),
    ((1024, 2048), [1024, 1280, 1536, 1792, 2048]),
    ((1, 8, 64), [1, 8, 64]),          # a thin list stays as it is
    ((1, 1024), [1, 1024]),
    ((256, 300), [256, 300]),
    ((7,), [7]),
])
def test_fill_buckets(listed, want):
    assert fill_buckets(listed) == want


def test_fill_buckets_waste():
    """From 33 rows on, a step computes at most a third of padding, and the listed sizes are all there."""
    sizes = fill_buckets(LISTED)
    assert set(LISTED) <= set(sizes) and sizes == sorted(set(sizes))
    for n in range(33, LISTED[-1] + 1):
        b = next(b for b in sizes if b >= n)
        assert b - n < max(16, n // 3)


@pytest.mark.gpu
@pytest.mark.parametrize("model", ["llama3-8b", "mixtral-8x7b"])
@pytest.mark.parametrize("n", [33, 81, 129, 193, 257, 321])
def test_step_in_an_added_size(gpu, model, n):
    """Full width, two layers: logits of a decode step in a graph of 48 .. 384 rows against the eager step of the same
    sequences.  Tiles and K ranges differ between the two, so every bf16 activation may round the other way: two layers'
    activations are rounded about a dozen times at 2^-9 each, 0.4 % * sqrt(12) = 1.4 % at most of each row; four times that."""
    cfg = get_config(model, num_layers=2)
    torch.manual_seed(0)
    m = build_model(cfg, device=gpu, seed=1)
    if cfg.num_experts:  # the experts' choice is a discontinuity: let it be clear
        for L in m.layers:
            L["router"].mul_(8)
    toks = torch.randint(10, cfg.vocab_size - 10, (n, 4), generator=torch.Generator().manual_seed(n)).tolist()
    out = []
    for graphs in (True, False):
        eng = Engine(m, EngineConfig(max_num_seqs=512, max_num_batched_tokens=2048, max_model_len=256, num_kv_blocks=n + 8,
                                     use_graphs=graphs, graph_buckets=(32, 64, 128, 256, 512), enable_prefix_caching=False))
        seqs = [eng.open_sequence() for _ in range(n)]
        eng.feed([(s, t[:3], []) for s, t in zip(seqs, toks)])
        if graphs:
            assert n not in eng.graphs and min(b for b in eng.graphs if b >= n) < n + 64
        out.append(eng.feed([(s, t[3:], [0]) for s, t in zip(seqs, toks)]).float())
        assert out[-1].shape == (n, cfg.vocab_size) and bool(torch.isfinite(out[-1]).all())
    a, b = out
    rows = ((a - b).norm(dim=1) / b.norm(dim=1)).sort().values
    # a token whose second and third expert are level may go either way (mixtral): all rows but one in twenty
    assert float(rows[int(len(rows) * 0.95) if cfg.num_experts else -1]) < 0.06


@pytest.mark.gpu
@pytest.mark.parametrize("model", ["llama3-8b", "llama3-70b"])
def test_added_size_keeps_the_norm_chain(gpu, model):
    """Where the listed graph has the norm chain (row factors in 32 bits on the accumulators, sums into the residual), every
    added size below it has it too: a step is not rounded once more because it runs in fewer rows."""
    m = build_model(get_config(model, num_layers=1), device=gpu, seed=1)
    rows, layer = set(), m._chain_layer

    def spy(i, a, *args):
        rows.add(a.shape[0])
        return layer(i, a, *args)

    m._chain_layer = spy
    eng = Engine(m, EngineConfig(max_num_seqs=1024, max_num_batched_tokens=2048, max_model_len=256, num_kv_blocks=64))
    assert 1024 in rows and set(eng.graphs) == set(fill_buckets(LISTED))
    for b in eng.graphs:
        assert b in rows or next(n for n in LISTED if n >= b) not in rows, (b, sorted(rows))


@pytest.mark.gpu
@pytest.mark.parametrize("model", ["llama3-8b", "mixtral-8x7b"])
def test_added_sizes_are_not_run_before_their_capture(gpu, model):
    """An engine starts with one run of the model per listed size; the added ones are captured only."""
    m = build_model(get_config(model, num_layers=1), device=gpu, seed=1)
    ran, caught, forward = [], [], m.forward

    def spy(ids, *args):
        (caught if torch.cuda.is_current_stream_capturing() else ran).append(ids.shape[0])
        return forward(ids, *args)

    m.forward = spy
    Engine(m, EngineConfig(max_num_seqs=512, max_num_batched_tokens=2048, max_model_len=256, num_kv_blocks=64))
    listed = [b for b in LISTED if b <= 512]
    assert sorted(ran) == listed and sorted(caught) == fill_buckets(listed)
