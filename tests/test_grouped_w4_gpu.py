"""The experts' products on four-wave tiles (gemm_w4_grouped_kernel, gate_up of prompts) against fp32: routings that
lead to each tile height, empty and full experts, gathered rows, every epilogue, with and without the K-half tail."""
import pytest
import torch

from mlopamd import ops

pytestmark = pytest.mark.gpu
bf = torch.bfloat16
G, N = 8, 24576

COUNTS = {
    "even-150": [150] * G,  # one tile of 160 rows each
    "one-row-over": [161, 193, 257, 160, 192, 256, 1, 0],
    "one-expert": [0, 0, 0, 0, 0, 0, 0, 613],
    "first-and-last": [257, 0, 0, 0, 0, 0, 0, 300],
    "even-190": [190] * G,
    "even-250": [250, 256, 249, 255, 251, 256, 240, 256],
    "skewed": [1500, 3, 17, 0, 64, 5, 90, 700],
    "single-row": [0, 0, 0, 1, 0, 0, 0, 0],
    "even-224": [224] * G,
    "even-448": [448] * G,
    "seven-448": [448] * 7 + [0],
    "224-edges": [223, 0, 447, 225, 448, 449, 672, 0],
    "above-512-each": [0, 896, 224, 672, 896, 1120, 0, 672],  # the K walk of larger prompts
}
# the height that each leads to at K = 192 / 448 / 1536, and whether its tail is cut into K-halves there
HEIGHTS = {
    "even-150": ("160", "160", "160"),
    "one-row-over": ("256", "256", "256"),
    "one-expert": ("160", "160", "160 halves"),
    "first-and-last": ("160", "160", "160 halves"),
    "even-190": ("192", "192", "192"),
    "even-250": ("256", "256", "256"),
    "skewed": ("224", "224", "192 halves"),
    "single-row": ("160", "160", "160 halves"),
    "even-224": ("224", "224", "224"),
    "even-448": ("224", "224", "224"),
    "seven-448": ("224", "224", "224 halves"),
    "224-edges": ("224", "224", "224"),
    "above-512-each": ("224", "224", "224 halves"),
}


def glu(z, lim):
    g, u = ops.deinterleave_cols(z).chunk(2, -1)
    if lim is None:
        return g, u, g * g.sigmoid() * u
    gc, uc = g.clamp(max=lim[1]), u.clamp(-lim[1], lim[1])
    return gc, uc + 1, gc * (lim[0] * gc).sigmoid() * (uc + 1)


@pytest.mark.parametrize("name", COUNTS)
def test_heights(gpu, name):
    """Each routing leads to the height it stands for, and all four are there, with K-halves where a height may have them."""
    cus, got = torch.cuda.get_device_properties(gpu).multi_processor_count, []
    for K in (192, 448, 1536):
        h = torch.ops.mlop.gemm_grouped_height(COUNTS[name], N, K, cus)
        tail = sum(-(-c // h) for c in COUNTS[name]) * (N // 256) % cus
        got.append(f"{h} halves" if K // 64 % 2 == 0 and 0 < 2 * tail <= cus else str(h))
    assert tuple(got) == HEIGHTS[name]


@pytest.mark.parametrize("counts", COUNTS.values(), ids=COUNTS.keys())
@pytest.mark.parametrize("K", [192, 448, 1536])
@pytest.mark.parametrize("kind", ["plain", "silu", "gathered", "scaled", "clamped"])
def test_grouped(gpu, counts, K, kind):
    torch.manual_seed(K + sum(counts))
    off = torch.tensor([0] + counts, device=gpu).cumsum(0).int()
    R = int(off[-1])
    w = 0.05 * torch.randn(G, N, K, device=gpu, dtype=bf)
    gather = kind not in ("plain", "silu")
    toks = torch.randn(R // 2 + 1 if gather else R, K, device=gpu, dtype=bf)
    rows = torch.randint(0, toks.shape[0], (R,), device=gpu, dtype=torch.int32) if gather else None
    scale = 0.5 + torch.rand(R, device=gpu) if kind == "scaled" else None
    lim = (1.702, 3.0) if kind == "clamped" else None
    epi = 0 if kind == "plain" else 1
    ops._sk_reserve(torch.device(gpu))
    assert torch.ops.mlop.gemm_grouped_variant(R, N, K, G, 64, toks.shape[0]) == 5
    got = [ops.grouped_gemm(toks, w, off, epi=epi, avg_rows=64, a_rows=rows,
                            row_scale=scale, glu=lim) for _ in range(8)]
    assert all(torch.equal(got[0], g) for g in got[1:])
    x = toks[rows.long()] if gather else toks
    for e in range(G):
        a, b = int(off[e]), int(off[e + 1])
        if a == b:
            continue
        xe, we = x[a:b].float(), w[e].float()
        y, sums = xe @ we.t(), 2.0 ** -20 * (xe.abs() @ we.abs().t())  # fp32 sums in another order
        if scale is not None:
            y, sums = y * scale[a:b, None], sums * scale[a:b, None]
        if epi == 0:
            exp, bound = y, 2.0 ** -8 * y.abs() + 2 * sums
        else:  # roundings of gate, up, the gated half and the product; |d (g sigmoid) / dg| <= 1.1
            g, u, exp = glu(y, lim)
            sg, su = ops.deinterleave_cols(sums).chunk(2, -1)
            bound = 4 * 2.0 ** -8 * g.abs() * (u.abs() + (lim is not None)) + 1.1 * sg * u.abs() + su * g.abs()
        assert ((got[0][a:b].float() - exp).abs() <= bound + 1e-5).all(), e


@pytest.mark.parametrize("height,counts", [(160, [150, 159, 160, 145, 152, 140, 151, 129]), (192, [190, 161, 192, 185, 177, 129, 191, 170]),
                                           (224, [430, 448, 440, 225, 400, 448, 410, 390]), (256, [257, 10, 300, 255, 250, 256, 240, 256])])
@pytest.mark.parametrize("gather", [False, True])
@pytest.mark.parametrize("epi", [0, 1])
def test_rows_past_an_experts_last(gpu, height, counts, gather, epi):
    """They load nothing: what the LDS holds there (a product of NaN before) reaches no output, and the waits that count the
    dropped loads cover the others, the next tile's among them (three tiles a workgroup and more): bit for bit what the same rows give
    in as many tiles without a partial one."""
    K, cus = 448, torch.cuda.get_device_properties(gpu).multi_processor_count
    full = [-(-c // height) * height for c in counts]
    assert all(torch.ops.mlop.gemm_grouped_height(c, N, K, cus) == height for c in (counts, full))
    torch.manual_seed(height)
    w = 0.05 * torch.randn(G, N, K, device=gpu, dtype=bf)
    ends = lambda c: torch.tensor([0] + c, device=gpu).cumsum(0).int()  # noqa: E731
    off, off_full = ends(counts), ends(full)
    toks = torch.randn(int(off[-1]), K, device=gpu, dtype=bf)
    rows = torch.randperm(toks.shape[0], device=gpu).int() if gather else None
    x = toks[rows.long()] if gather else toks
    at = torch.cat([torch.arange(c, device=gpu) + int(off_full[e]) for e, c in enumerate(counts)])
    padded = torch.randn(sum(full), K, device=gpu, dtype=bf)
    padded[at] = x
    ops._sk_reserve(torch.device(gpu))
    want = ops.grouped_gemm(padded, w, off_full, epi=epi, avg_rows=64)[at]
    nan, nan_off = torch.full((G * 448, K), float("nan"), device=gpu, dtype=bf), ends([448] * G)
    for _ in range(4):
        ops.grouped_gemm(nan, w, nan_off, epi=epi, avg_rows=64)
        assert torch.equal(ops.grouped_gemm(toks, w, off, epi=epi, avg_rows=64, a_rows=rows), want)
