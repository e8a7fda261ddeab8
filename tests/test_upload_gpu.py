"""The step's upload kernel: runs and a block of pinned host words to the same places on the device, nothing else."""
import pytest
import torch

from mlopamd.runtime.attn_meta import MetaBuffers

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("runs,block", [([(0, 2)], (0, 0, 0, 0)), ([(16, 2), (64, 510), (640, 514)], (3, 6, 10, 2000)),
                                        ([], (1, 2, 2, 4094)), ([(0, 4096)], (0, 4, 8, 0)), ([(i * 64, 62) for i in range(12)], (700, 4, 4, 1024))])
def test_words(gpu, runs, block):
    n = 4096
    src = torch.arange(1, n + 1, dtype=torch.int32).pin_memory()
    dst = torch.zeros(n, dtype=torch.int32, device=gpu)
    exp = torch.zeros(n, dtype=torch.int32)
    for o, c in runs:
        exp[o:o + c] = src[o:o + c]
    for r in range(block[0]):
        o = block[3] + r * block[2]
        exp[o:o + block[1]] = src[o:o + block[1]]
    flat = [x for p in runs for x in p] + list(block)
    torch.ops.mlop.upload(dst, src, flat)
    assert torch.equal(dst.cpu(), exp)
    src.neg_()  # rewritten by the host between two steps
    torch.ops.mlop.upload(dst, src, flat)
    assert torch.equal(dst.cpu(), -exp)


def test_refusals(gpu):
    src, dst = torch.zeros(256, dtype=torch.int32).pin_memory(), torch.zeros(256, dtype=torch.int32, device=gpu)
    for flat in ([0, 258, 0, 0, 0, 0], [1, 2, 0, 0, 0, 0], [-2, 2, 0, 0, 0, 0], [2, 8, 8, 256], [0, 2, 0, 0, 0], [2, 8, 4, 0]):
        with pytest.raises(RuntimeError):
            torch.ops.mlop.upload(dst, src, flat)


@pytest.mark.parametrize("tokens,seqs,rows_hi,ctx", [(64, 8, 3, 100), (33, 33, 33, 17), (1, 1, 1, 1), (64, 8, 0, 5), (50, 8, 8, 256)])
def test_step_arrays(gpu, tokens, seqs, rows_hi, ctx):
    """Everything a step of that many tokens reads is there; a second, smaller step too."""
    m = MetaBuffers(64, 64, 16, 4, 2, 256, gpu)
    g = torch.Generator().manual_seed(tokens + ctx)
    for T in (tokens, max(1, tokens // 2)):
        m.hbuf.random_(0, 1000, generator=g)
        m.view_h("ctx_len")[:] = ctx
        m.upload(T, min(T, seqs), rows_hi)
        h, d = m.hbuf, m.dbuf.cpu()
        for name in ("positions", "slots", "tile_seq", "tile_q0", "ptile_seq", "ptile_q0"):
            o = m.off[name][0]
            assert torch.equal(d[o:o + T], h[o:o + T]), name
        for name in ("q_start", "q_len", "ctx_len"):
            o, n = m.off[name]
            assert torch.equal(d[o:o + n], h[o:o + n]), name
        assert torch.equal(d[:m.HDR], h[:m.HDR]) and torch.equal(m.ids_d[:T].cpu(), m.ids_h[:T])
        assert torch.equal(m.lidx_d[:min(T, seqs)].cpu(), m.lidx_h[:min(T, seqs)])
        pages = -(-ctx // 16)
        assert torch.equal(m.view_d("block_tables").view(64, 16)[:rows_hi, :pages].cpu(), torch.from_numpy(m.bt_h[:rows_hi, :pages].copy()))
