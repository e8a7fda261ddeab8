"""Shares of a sequence's keys in decode attention (attention.hip even_parts / seq_part): launches of 72 to 376 (sequence, kv
head) pairs, two padding tiles among them, on either side of the lengths from which they are cut (376: of 888 keys on average),
alike and with one long sequence, with the host's sums of the lengths (AttnMeta.load) and without, combined in the launch and
by a second one."""
import numpy as np
import pytest
import torch

from mlopamd import ops
from mlopamd.runtime.attn_meta import MetaBuffers, plan_partitions

pytestmark = pytest.mark.gpu
bf = torch.bfloat16


@pytest.mark.parametrize("n,Hkv", [(9, 8), (17, 8), (33, 8), (47, 8), (72, 2), (160, 2)])
@pytest.mark.parametrize("ctx,longest", [(40, 40), (300, 0), (800, 0), (1300, 0), (200, 4000)])
def test_shares(gpu, n, Hkv, ctx, longest):
    G, D, mml, n = 4, 128, 4096, n - 2
    g = torch.Generator().manual_seed(n * ctx)
    c = (ctx * (0.75 + 0.5 * torch.rand(n, generator=g))).int().numpy()
    if longest:
        c[n // 2] = longest
    pages = [-(-int(x) // 16) for x in c]
    m = MetaBuffers(256, n + 3, mml // 16, G, Hkv, mml, gpu)
    perm = torch.randperm(sum(pages), generator=g).int().numpy()
    o = 0
    for i, p in enumerate(pages):
        m.bt_h[i, :p] = perm[o:o + p]
        o += p
    m.fill_decode(np.arange(n, dtype=np.int32), c, np.zeros(n, np.int64), pad_to=n + 2)
    m.upload()
    meta = m.meta(n + 2, n + 2, n + 2, *plan_partitions(n + 2, Hkv, mml))
    assert meta.load.tolist() == [int(c.sum()), n]
    k, v = (torch.randn(sum(pages) + 1, Hkv, 16, D, device=gpu, dtype=bf) for _ in range(2))
    q = torch.randn(n + 2, Hkv * G, D, device=gpu, dtype=bf)
    outs = [ops.paged_attention(q, k, v, meta)]
    meta.load = None
    outs.append(ops.paged_attention(q, k, v, meta))
    meta.part_sem = None
    outs.append(ops.paged_attention(q, k, v, meta))
    for i in range(n):
        rows = torch.as_tensor(m.bt_h[i, :pages[i]], device=gpu).long()
        kk, vv = (x[rows].transpose(1, 2).reshape(-1, Hkv, D)[:c[i]].double() for x in (k, v))
        s = torch.einsum("hgd,thd->hgt", q[i].double().view(Hkv, G, D), kk) * D ** -0.5
        e = torch.einsum("hgt,thd->hgd", s.softmax(-1), vv).reshape(Hkv * G, D)
        for out in outs:
            # weights are rounded to bf16 before the product (2^-9 of each, of values up to a few), the result once more
            assert float((out[i].double() - e).abs().max()) <= 2.0 ** -8 * float(e.abs().max()) + 2.0 ** -8, (i, int(c[i]))
    for out in outs:
        assert not bool(out[n:].any())
