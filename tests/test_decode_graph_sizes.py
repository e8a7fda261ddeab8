"""Decode graph sizes between the listed ones: which are added, and that a step in one of them gives what the
same step gives without graphs."""
import pytest
import torch

from mlopamd.models import build_model
from mlopamd.models.config import get_config
from mlopamd.runtime.engine import Engine, EngineConfig, fill_buckets
from mlopamd.runtime.sampler import SamplingParams

LISTED = EngineConfig.graph_buckets
BOUND = 0.032  # two layers in bf16, see test_step_in_an_added_size


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


@pytest.mark.parametrize("fill", [True, False])
def test_exactly_the_listed_sizes(fill):
    m = build_model(get_config("tiny-llama"), device="cpu", dtype=torch.float32)
    eng = Engine(m, EngineConfig(max_num_seqs=80, max_num_batched_tokens=128, max_model_len=64, num_kv_blocks=16,
                                 graph_buckets=(32, 64, 128), fill_graph_buckets=fill))
    assert eng.buckets == ([32, 48, 64, 80] if fill else [32, 64, 80])


@pytest.mark.gpu
@pytest.mark.parametrize("model", ["llama3-8b", "mixtral-8x7b"])
@pytest.mark.parametrize("n", [33, 81, 129, 193, 257, 321])
def test_step_in_an_added_size(gpu, model, n):
    """Full width, two layers: logits of a decode step in a graph of 48 .. 384 rows against the eager step of the same
    sequences.  Tiles and K ranges differ between the two, so every bf16 activation may round the other way.  A rounding is
    0.16 % of the value on average (2^-8 / sqrt(3) at a binade's lower end), two layers round about a dozen times, in two
    ways: 0.16 % * sqrt(2 * 12) = 0.8 % of a row; the bound is four times that."""
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
    assert float(rows[int(len(rows) * 0.95) if cfg.num_experts else -1]) < BOUND


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


HYBRID = ["kosesun-1b", "nafazen-1b", "dibedra-1b", "regesun-1b"]


def _spy_head(eng, m):
    """The head's calls: rows, whether a buffer was given, and the result of the scheduler's steps beside one in memory of its own."""
    calls, head, launch = [], m.logits_local, eng._launch

    def logits_local(hidden, out=None):
        calls.append((hidden.shape[0], out is not None))
        return head(hidden, out=out)

    def spy(kind, T, nt, nl, part, nparts, bucket, **kw):
        lg = launch(kind, T, nt, nl, part, nparts, bucket, **kw)
        if bucket:  # a graph's step
            steps.append((bucket, lg.data_ptr(), torch.equal(lg, head(eng._graph_hidden[bucket]))))
        return lg

    steps = []
    m.logits_local, eng._launch = logits_local, spy
    return calls, steps


@pytest.mark.gpu
@pytest.mark.parametrize("model", ["llama3-8b", "mixtral-8x7b", *HYBRID])
def test_graphs_share_one_logits_buffer(gpu, model):
    """The scheduler's steps of all sizes leave their logits in the buffer of the largest, and their graphs what the head reads in
    one other: the added sizes hold neither of their own."""
    m = build_model(get_config(model, num_layers=2), device=gpu, seed=1)
    eng = Engine(m, EngineConfig(max_num_seqs=128, max_num_batched_tokens=1024, max_model_len=256, num_kv_blocks=256))
    assert set(eng.graphs) == set(fill_buckets([b for b in LISTED if b <= 128]))
    assert len({h.data_ptr() for h in eng._graph_hidden.values()}) == 1
    assert all(h.shape[0] == b for b, h in eng._graph_hidden.items()) and eng._logits_buf.shape[0] == 128
    calls, steps = _spy_head(eng, m)
    long = {100: 3, 60: 6, 40: 9, 12: 12, 3: 15}  # sequences that go on for so many tokens: steps of 112, 64, 48, 16 and 4 rows
    n = [max(t for k, t in long.items() if i < k) for i in range(100)]
    eng.generate([[11 + i, 7, 5] for i in range(100)], [SamplingParams(max_tokens=t, ignore_eos=True) for t in n])
    assert {112, 64, 48, 16, 4} <= {b for b, _, _ in steps} and {a for _, a, _ in steps} == {eng._logits_buf.data_ptr()}
    assert all(same for _, _, same in steps)


@pytest.mark.gpu
@pytest.mark.parametrize("model,vocab", [("llama3-8b", None), ("dibedra-1b", None), ("kosesun-1b", 5001), ("regesun-1b", 5001)])
def test_what_feed_hands_out(gpu, model, vocab):
    """Logits that the caller keeps are written where it keeps them; not where they are not wanted, wanted in another order, or would
    hold far more than the wanted rows.  The values are those of the eager step, the tensor is dense, and holds little else."""
    m = build_model(get_config(model, num_layers=2, **({"vocab_size": vocab} if vocab else {})), device=gpu, seed=1)
    mk = lambda graphs: Engine(m, EngineConfig(max_num_seqs=128, max_num_batched_tokens=1024, max_model_len=256, num_kv_blocks=256,  # noqa: E731
                                               use_graphs=graphs, graph_buckets=(1, 16, 128), enable_prefix_caching=False))
    V, dense = m.cfg.vocab_size, not vocab  # (the head's rows are whole tiles)
    runs = []
    for graphs in (True, False):
        eng = mk(graphs)
        seqs = [eng.open_sequence() for _ in range(100)]
        eng.feed([(s, [11 + i, 7, 5], []) for i, s in enumerate(seqs)])
        if graphs:
            calls, _ = _spy_head(eng, m)
        out = []
        for rows, wanted in ((range(100), range(100)), (range(100), ()), (range(100), range(50)), (range(100), range(1, 100, 2)),
                             (range(12), range(12)), (range(20), range(20)), (range(1), range(1))):
            out.append(eng.feed([(seqs[i], [13 + i], [0] if i in wanted else []) for i in rows]))
            if graphs:
                assert len(calls) == 1
                calls.clear() if out[-1] is None else out.append(calls.pop())
        torch.cuda.synchronize()
        runs.append(out)
        if graphs:
            del m.logits_local
    got, buffered = [x for x in runs[0] if not isinstance(x, tuple)], [x[1] for x in runs[0] if isinstance(x, tuple)]
    # (all, none, half, every second, 12 in 16 rows, 20 in 128, 1)
    assert buffered == ([False, True, True, False, True, False] if dense else [True] * 6)
    for a, b in zip(got, runs[1]):
        assert (a is None) == (b is None)
        if a is not None:
            assert a.is_contiguous() and a.dtype == b.dtype and a.shape == b.shape == (a.shape[0], V)
            assert a.untyped_storage().nbytes() <= max(4 * a.numel() // 3, a.numel() + 32 * V) * a.element_size()
            assert float(_row_errors(a.float(), b.float())[-1]) < BOUND


def _steps(m, n, graphs, steps, listed=LISTED, rows=512):
    """Logits of the decode steps over ``steps`` sequences each (a prefix of n sequences of three tokens), all kept until the
    last one ran; and the engine."""
    toks = torch.randint(10, m.cfg.vocab_size - 10, (n, 3 + len(steps)), generator=torch.Generator().manual_seed(n)).tolist()
    eng = Engine(m, EngineConfig(max_num_seqs=rows, max_num_batched_tokens=max(2048, 3 * n), max_model_len=256,
                                 num_kv_blocks=n + 8, use_graphs=graphs, graph_buckets=listed, enable_prefix_caching=False))
    seqs = [eng.open_sequence() for _ in range(n)]
    eng.feed([(s, t[:3], []) for s, t in zip(seqs, toks)])
    out = [eng.feed([(s, [t[3 + i]], [0]) for s, t in zip(seqs[:k], toks)]) for i, k in enumerate(steps)]
    torch.cuda.synchronize()
    return [o.float() for o in out], eng


def _row_errors(a, b):
    return ((a - b).norm(dim=1) / b.norm(dim=1)).sort().values


@pytest.mark.gpu
@pytest.mark.parametrize("model", HYBRID)
@pytest.mark.parametrize("n", [33, 81, 193, 321])
def test_hybrid_step_in_an_added_size(gpu, model, n):
    """The models with recurrent layers, four layers of them; the same steps with and without graphs, twice one after the
    other (the second reads the state that the first left)."""
    m = build_model(get_config(model, num_layers=4), device=gpu, seed=1)
    got, eng = _steps(m, n, True, [n, n])
    want, _ = _steps(m, n, False, [n, n])
    assert min(g for g in eng.graphs if g >= n) not in LISTED
    for a, b in zip(got, want):
        assert a.shape == (n, m.cfg.vocab_size) and bool(torch.isfinite(a).all())
        # twice the layers of BOUND; a token whose experts are level may go either way
        assert float(_row_errors(a, b)[int(n * 0.95)]) < 2 ** 0.5 * BOUND


@pytest.mark.gpu
@pytest.mark.parametrize("model", ["llama3-8b", "mixtral-8x7b"])
@pytest.mark.parametrize("n", [385, 577, 705, 833, 1025, 1537])
def test_step_in_a_large_added_size(gpu, model, n):
    """The steps of 64 and of 256 rows, as test_step_in_an_added_size."""
    m = build_model(get_config(model, num_layers=2), device=gpu, seed=1)
    if m.cfg.num_experts:
        for L in m.layers:
            L["router"].mul_(8)
    (a,), eng = _steps(m, n, True, [n], (*LISTED, 2048), 2048)
    (b,), _ = _steps(m, n, False, [n], (*LISTED, 2048), 2048)
    assert min(g for g in eng.graphs if g >= n) not in (*LISTED, 2048)
    assert float(_row_errors(a, b)[int(n * 0.95) if m.cfg.num_experts else -1]) < BOUND


@pytest.mark.gpu
@pytest.mark.parametrize("model", ["llama3-8b", "kosesun-1b"])
def test_logits_outlive_the_next_step(gpu, model):
    """What ``feed`` returned stays as it was while steps of other sizes run, whether the head wrote it there or it is a copy of the
    graphs' one buffer."""
    m = build_model(get_config(model, num_layers=2), device=gpu, seed=1)
    steps = [90, 40, 90, 7]
    got, eng = _steps(m, 90, True, steps)
    want, _ = _steps(m, 90, False, steps)
    assert {min(g for g in eng.graphs if g >= k) for k in steps} == {96, 48, 8}
    for k, a, b in zip(steps, got, want):
        assert a.shape[0] == k and float(_row_errors(a, b)[-1]) < BOUND
