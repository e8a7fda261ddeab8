"""Flash prefill (attention.hip flash_item) where its pipeline begins and ends: one pair of pages up to more than two rounds
of its unrolled loop, last pairs of one key to 32, rows that move the running max at every pair."""
import numpy as np
import pytest
import torch

from mlopamd import ops
from mlopamd.ops import reference as ref

pytestmark = pytest.mark.gpu
bf = torch.bfloat16


def launch(gpu, q_lens, ctx_lens, Hq, Hkv, grow, keys=0, spoil=None):
    """Every sequence a prefill of q_lens tokens behind ctx_lens - q_lens cached ones, pages scattered.  spoil(q, k_cache,
    v_cache, block tables) puts values there that the reference is not compared with."""
    G, rng, S = Hq // Hkv, np.random.default_rng(len(q_lens) + Hq), len(q_lens)
    pages = [(c + 15) // 16 for c in ctx_lens]
    NB = sum(pages) + 3
    ids = rng.permutation(np.arange(1, NB))
    bt = np.zeros((S, max(pages)), np.int32)
    seq, q0 = [], []
    for i, n in enumerate(pages):
        bt[i, :n] = ids[sum(pages[:i]):sum(pages[:i]) + n]
        first = list(range(0, q_lens[i], 128 // G))
        seq += [i] * len(first)
        q0 += first[::-1]

    class Meta:
        pass

    m, d = Meta(), lambda a: torch.tensor(np.asarray(a), dtype=torch.int32, device=gpu)
    m.block_tables, m.ctx_len, m.q_len = d(bt), d(ctx_lens), d(q_lens)
    m.q_start = d(np.concatenate([[0], np.cumsum(q_lens)[:-1]]))
    m.tile_seq = m.tile_q0 = d(np.zeros(0))
    m.ptile_seq, m.ptile_q0 = d(seq), d(q0)
    m.part_tokens, m.nparts = max(ctx_lens), 1
    m.part_o = m.part_ml = torch.empty(1, device=gpu)
    torch.manual_seed(S)
    q = torch.randn(sum(q_lens), Hq, 128, device=gpu, dtype=bf)
    kc, vc = (torch.randn(NB, Hkv, 16, 128, device=gpu, dtype=bf) for _ in range(2))
    if grow:  # larger keys the later they stand
        for i, n in enumerate(pages):
            at = torch.arange(n, device=gpu).view(n, 1, 1, 1)
            kc[bt[i, :n]] = (kc[bt[i, :n]].float() * 1.25 ** (at % 24)).to(bf)
    m.pkeys = keys
    if spoil is not None:
        spoil(q, kc, vc, bt)
        return ops.paged_attention(q, kc, vc, m)
    out = ops.paged_attention(q, kc, vc, m)
    exp = ref.paged_attention(q, kc, vc, m)
    # P in bf16 (2^-9 of each addend, which the row's sum does not share) and the result's rounding; |V| < 5
    torch.testing.assert_close(out.float(), exp.float(), atol=2.0 ** -6, rtol=2.0 ** -6)
    return out, lambda: ops.paged_attention(q, kc, vc, m)


@pytest.mark.parametrize("grow", [False, True])
@pytest.mark.parametrize("Hq,Hkv", [(8, 8), (8, 2), (16, 2)])
def test_every_number_of_pairs(gpu, Hq, Hkv, grow):
    ctx = [32 * p + r for p in range(14) for r in (1, 16, 17, 32)]
    launch(gpu, [min(c, 1 + 7 * i % 23) for i, c in enumerate(ctx)], ctx, Hq, Hkv, grow)


@pytest.mark.parametrize("Hq,Hkv", [(8, 8), (8, 2), (16, 2)])
def test_whole_prompts(gpu, Hq, Hkv):
    n = [1, 15, 31, 32, 33, 63, 64, 65, 97, 127, 128, 129, 190, 255, 257, 449]
    launch(gpu, n, n, Hq, Hkv, False)


@pytest.fixture
def in_turn(gpu):
    torch.ops.mlop.flash_form(2)
    yield
    torch.ops.mlop.flash_form(0)


@pytest.mark.parametrize("grow", [False, True])
@pytest.mark.parametrize("Hq,Hkv", [(8, 8), (8, 4), (8, 2), (16, 2)])
def test_in_turn(gpu, in_turn, Hq, Hkv, grow):
    """The form of short tiles, whose rings are three pairs deep, over the same numbers of pairs and lengths."""
    ctx = [32 * p + r for p in range(11) for r in (1, 16, 17, 32)]
    launch(gpu, [min(c, 1 + 7 * i % 23) for i, c in enumerate(ctx)], ctx, Hq, Hkv, grow)
    n = [1, 15, 31, 32, 33, 63, 64, 65, 97, 127, 128, 129, 190, 255, 257, 449]
    launch(gpu, n, n, Hq, Hkv, grow)


@pytest.mark.parametrize("tiles,mean,turn", [(28, 80, True), (28, 81, False), (29, 20, False), (64, 20, False), (65, 20, True), (80, 180, True), (80, 181, False),
                                             (112, 256, True), (113, 20, False), (128, 20, False), (129, 200, True), (129, 202, False), (400, 512, True), (400, 513, False)])
def test_which_form(gpu, tiles, mean, turn):
    """8 kv heads, short prompts of one tile each: the form that the rule names, bit for bit (the two sum in other orders)."""
    out, again = launch(gpu, [1 + i % 16 for i in range(tiles)], [100 + i for i in range(tiles)], 64, 8, False, keys=tiles * mean)
    try:
        torch.ops.mlop.flash_form(2 if turn else 1)
        assert torch.equal(out, again())
        torch.ops.mlop.flash_form(1 if turn else 2)
        assert not torch.equal(out, again())
    finally:
        torch.ops.mlop.flash_form(0)


@pytest.mark.parametrize("grow", [False, True])
@pytest.mark.parametrize("Hq,Hkv", [(2, 2), (4, 2), (8, 2), (16, 2)])
@pytest.mark.parametrize("pairs", [30, 60, 120, 1000])
def test_key_ranges(gpu, Hq, Hkv, grow, pairs):
    """A tile's keys in ranges, merged: of a pair and of many, tiles with fewer pairs than ranges beside long ones, ranges that
    end in the tile's diagonal (rows whose keys all lie before the last ones), uneven ones."""
    q = [37, 1, 50, 33, 5]
    tiles = sum(-(-n // (128 * Hkv // Hq)) for n in q)
    splits = torch.ops.mlop.flash_splits(tiles, Hkv, tiles * 32 * pairs)  # (11 - 16; the launch does with what it is told)
    assert splits > 4
    ctx = [37, 33, 32 * splits + 1, 1500, 32 * 41 + 5]
    out, again = launch(gpu, q, ctx, Hq, Hkv, grow, keys=tiles * 32 * pairs)
    assert torch.equal(out, again())
    whole, _ = launch(gpu, q, ctx, Hq, Hkv, grow)
    # both P in bf16 against another max (2^-9 of each addend) and rounded
    torch.testing.assert_close(out.float(), whole.float(), atol=2.0 ** -7, rtol=2.0 ** -7)


def spoil_key(q, kc, vc, bt, at=777):
    kc[bt[1, at // 16], :, at % 16, 5] = float("nan")


def spoil_query(q, kc, vc, bt):
    q[40, 1, 7] = float("nan")


def spoil_score(q, kc, vc, bt, at=777):
    """One key whose scores are +infinity for some rows and, as good as -infinity or masked by it, nothing for others."""
    kc[bt[1, at // 16], :, at % 16] = 0
    kc[bt[1, at // 16], :, at % 16, 5] = 3e38
    q[..., 5] = torch.where(q[..., 5] >= 0, 2.0, -2.0).to(bf)


def spoil_values(q, kc, vc, bt):
    vc[bt[1, 3], :, 4, 100], vc[bt[1, 80], :, 2, 3] = float("nan"), float("inf")


@pytest.mark.parametrize("Hq,Hkv", [(2, 2), (8, 2)])
@pytest.mark.parametrize("spoil", [spoil_key, spoil_query, spoil_score, spoil_values, lambda *a: [spoil_key(*a, at=i) for i in range(0, 1500, 7)]],
                         ids=["key", "query", "score", "values", "keys"])
def test_key_ranges_of_what_is_not_finite(gpu, spoil, Hq, Hkv):
    """A NaN or an infinity shows in the same outputs as without ranges: of a range that holds it no row is dropped."""
    q, ctx = [37, 50, 5], [1500, 1500, 900]
    tiles = sum(-(-n // (128 * Hkv // Hq)) for n in q)
    keys = tiles * 32 * 60
    assert torch.ops.mlop.flash_splits(tiles, Hkv, keys) > 4
    got, whole = (launch(gpu, q, ctx, Hq, Hkv, False, keys=k, spoil=spoil).float() for k in (keys, 0))
    assert not torch.isfinite(whole).all() and torch.isfinite(whole).any()
    torch.testing.assert_close(got, whole, atol=2.0 ** -7, rtol=2.0 ** -7, equal_nan=True)


@pytest.mark.parametrize("q,cached,splits", [(417, 2000, 4), (417, 1000, 2), (800, 4000, 2), (150, 700, 6), (150, 400, 5)])
def test_key_ranges_of_chunks(gpu, q, cached, splits):
    keys = sum(min(q, a + 32) + cached for a in range(0, q, 32))
    assert torch.ops.mlop.flash_splits(-(-q // 32), 8, keys) == splits
    launch(gpu, [q], [q + cached], 32, 8, False, keys=keys)


def test_key_ranges_rule(gpu):
    f = torch.ops.mlop.flash_splits
    assert f(5, 8, 0) == f(5, 8, 5 * 150) == f(29, 8, 29 * 250) == f(128, 8, 128 * 11000) == 1  # unknown, short, many workgroups
    assert f(5, 8, 5 * 4000) > 1 and f(16, 8, 16 * 12000) > 1
    assert all(t * h * f(t, h, t * k) <= 512 or f(t, h, t * k) == 1 for t in (1, 3, 17, 40, 65) for h in (1, 2, 8, 32) for k in (100, 3000, 90000))
