"""Engine steps that a predictor of this package runs while it serves: decode batches, prompts, chunks of long prompts
and steps that hold both, on the dense and the expert model families.

A case is one step of ``Engine.feed`` over given tokens: ``decode`` sequences of about ``ctx`` tokens that get one
token each, beside ``prompts`` portions of about ``prompt`` tokens behind ``cached`` earlier ones.  Lengths are spread
a quarter to either side of these means, as a batch's are.  The models are the presets' with fewer layers (a state has
its own weights, pages and captured graphs), random weights of the presets' scale, bf16, the type that is served.
After a pass the sequences are set back to where they were: the next pass feeds the same positions again.
"""
from __future__ import annotations

import math

import torch

from mlopamd import ops
from mlopamd.models import build_model
from mlopamd.models.config import get_config
from mlopamd.runtime.engine import Engine, EngineConfig
from mlopamd.runtime.kv_cache import BLOCK_SIZE

LAYERS = {"llama3-8b": 6, "llama3-70b": 3, "mixtral-8x7b": 3}
KEYS = {"llama3-8b": 360_000, "llama3-70b": 120_000, "mixtral-8x7b": 200_000}   # drawn steps: keys in the pages
TOKENS = {"llama3-8b": 8192, "llama3-70b": 3072, "mixtral-8x7b": 6144}          # and tokens fed
STEP = 8192     # tokens of one engine step
TEXTS = 4       # sequences begin with one of so many texts (one where contexts are long)


def _case(name, model, decode=0, ctx=0, prompts=0, prompt=0, cached=0):
    d = {"model": model, "decode": decode, "ctx": ctx, "prompts": prompts, "prompt": prompt, "cached": cached}
    return {"name": name, **d} if name else d


def listed():
    return [
        # one user's tokens, one after the other: launches and one pass over the weights
        _case("decode-1", "llama3-8b", decode=1, ctx=900),
        # a quiet predictor: a handful of conversations
        _case("decode-13", "llama3-8b", decode=13, ctx=2500),
        # few users with documents in context: the pages are what is read
        _case("decode-3-long", "llama3-8b", decode=3, ctx=24000),
        # a busy one, no power of two
        _case("decode-100", "llama3-8b", decode=100, ctx=1000),
        # the throughput end of continuous batching
        _case("decode-700", "llama3-8b", decode=700, ctx=500),
        # a chat turn read at once
        _case("prompt-150", "llama3-8b", prompts=1, prompt=150),
        # a few prompts that arrived together
        _case("prompt-3x333", "llama3-8b", prompts=3, prompt=333),
        # an offline batch's prompts, a whole step
        _case("prompt-16x500", "llama3-8b", prompts=16, prompt=500),
        # prompts read beside running sequences (the engine's mixed step)
        _case("mixed-300-5x400", "llama3-8b", decode=300, ctx=600, prompts=5, prompt=400),
        # the wide model, a chunk of a long document
        _case("chunk-70b", "llama3-70b", prompts=1, prompt=2048, cached=9000),
        # experts: a decode batch, and prompts
        _case("experts-decode-20", "mixtral-8x7b", decode=20, ctx=800),
        _case("experts-prompt-2x900", "mixtral-8x7b", prompts=2, prompt=900),
    ]


def _between(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    model = rng.choice(["llama3-8b"] * 4 + ["mixtral-8x7b"] * 2 + ["llama3-70b"])
    kind = rng.choice(["decode"] * 4 + ["prompt"] * 3 + ["chunk", "mixed"])
    decode = ctx = prompts = prompt = cached = 0
    if kind in ("decode", "mixed"):
        decode = _between(rng, 1, 1000)
        ctx = _between(rng, 64, max(64, min(24000, KEYS[model] // decode)))
    if kind != "decode":
        room = TOKENS[model] - decode
        prompts = 1 if kind == "chunk" else _between(rng, 1, 16)
        prompt = _between(rng, 16, max(16, min(6000, room * 3 // 4 // prompts)))
        cached = _between(rng, 256, 12000) if kind == "chunk" else 0
    return _case(None, model, decode, ctx, prompts, prompt, cached)


# ---------------------------------------------------------------- shapes --

def _spread(n, mean):
    """n lengths about ``mean``, from three quarters to five quarters of it."""
    return [mean] if n == 1 else [max(1, int(mean * (0.75 + 0.5 * (i * 0.6180339887 % 1.0)))) for i in range(n)]


def _sequences(case):
    """(tokens before the step, tokens fed) of each sequence."""
    return ([(c - 1, 1) for c in (max(2, c) for c in _spread(case["decode"], case["ctx"]))]
            + [(case["cached"], max(2, t)) for t in _spread(case["prompts"], case["prompt"])])


def _config(case):
    longest = max(c + t for c, t in _sequences(case))
    return get_config(case["model"], num_layers=LAYERS[case["model"]], max_position=max(8192, 1 << (longest + 15).bit_length()))


def _keys(case):
    """Keys that the queries of a step meet, over all sequences."""
    return sum(t * c + t * (t + 1) // 2 for c, t in _sequences(case))


def work(case):
    cfg, seqs = _config(case), _sequences(case)
    H, I, L, V = cfg.hidden_size, cfg.intermediate_size, cfg.num_layers, cfg.vocab_size
    q, kv = cfg.num_heads * cfg.head_dim, cfg.num_kv_heads * cfg.head_dim
    T, n = sum(t for _, t in seqs), len(seqs)
    attn, mlp = H * (q + 2 * kv) + H * q, 3 * H * I
    if cfg.num_experts:
        read = cfg.num_experts * (1 - (1 - cfg.top_k / cfg.num_experts) ** T)  # experts that some token chose, on average
        weights, per_token = attn + read * mlp + cfg.num_experts * H, attn + cfg.top_k * mlp + cfg.num_experts * H
    else:
        weights = per_token = attn + mlp
    pages = sum(c + 2 * t for c, t in seqs) * 2 * kv  # earlier keys and values read, new ones written and read
    return {"bytes": 2 * (L * (weights + pages) + V * H + T * H + n * V),
            "flops": 2.0 * (T * L * per_token + n * V * H) + 4.0 * q * L * _keys(case)}


# ------------------------------------------------------- weights, tokens --

def _weights(cfg, seed):
    """The model's tensors in order: ("embed", ...), (i, {...}) per layer, ("lm_head", ...)."""
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)

    def w(*shape):
        return torch.empty(*shape, device="cuda", dtype=torch.bfloat16).normal_(0.0, 0.02, generator=gen)

    H, I, V, E = cfg.hidden_size, cfg.intermediate_size, cfg.vocab_size, cfg.num_experts
    q, kv = cfg.num_heads * cfg.head_dim, cfg.num_kv_heads * cfg.head_dim
    embed = w(V, H)
    if E:
        # Which experts a token gets is a discontinuity.  A trained router's choice is the token's; here E coordinates
        # of the residual stream hold it (two of them set, the rest zero) and nothing else writes to them.
        pick = torch.rand(V, E, device="cuda", generator=gen).topk(2, dim=1).indices
        embed[:, :E] = 0
        embed[:, :E].scatter_(1, pick, torch.tensor([0.32, 0.25], device="cuda", dtype=embed.dtype).expand(V, 2))
    yield "embed", embed
    for i in range(cfg.num_layers):
        d = {"q": w(q, H), "k": w(kv, H), "v": w(kv, H), "o": w(H, q)}
        if E:
            d["o"][:E] = 0
            d["router"] = torch.zeros(E, H, device="cuda", dtype=torch.bfloat16)
            d["router"][torch.arange(E), (torch.arange(E) + i) % E] = 1.5
            d["gate"], d["up"], d["down"] = w(E, I, H), w(E, I, H), w(E, H, I)
            d["down"][:, :E] = 0
        else:
            d["gate"], d["up"], d["down"] = w(I, H), w(I, H), w(H, I)
        yield i, d
    yield "lm_head", w(V, H)


def _tokens(case, cfg, seed):
    """(texts that sequences begin with, index of each sequence's text, tokens fed to each)."""
    seqs = _sequences(case)
    g = torch.Generator().manual_seed(seed)
    before = max(c for c, _ in seqs)
    texts = torch.randint(10, cfg.vocab_size - 10, (TEXTS if before <= 4096 else 1, before), generator=g).tolist()
    fed = [torch.randint(10, cfg.vocab_size - 10, (t,), generator=g).tolist() for _, t in seqs]
    return texts, [i % len(texts) for i in range(len(seqs))], fed


# ------------------------------------------------------------------ run --

def prepare(case, seed):
    cfg, seqs = _config(case), _sequences(case)
    model = build_model(cfg, device="cuda")
    for at, w in _weights(cfg, seed):
        if at == "embed":
            model.embed.copy_(w)
        elif at == "lm_head":
            model.lm_head.copy_(w)
        else:
            L = model.layers[at]
            L["qkv"].copy_(torch.cat([w["q"], w["k"], w["v"]]))
            L["o"].copy_(w["o"])
            if cfg.num_experts:
                L["router"].copy_(w["router"])
                for e in range(cfg.num_experts):
                    L["w13"][e].copy_(ops.interleave_gate_up(w["gate"][e], w["up"][e]))
                L["w2"].copy_(w["down"])
            else:
                L["gate_up"].copy_(ops.interleave_gate_up(w["gate"], w["up"]))
                L["down"].copy_(w["down"])
    longest = max(c + t for c, t in seqs) + 16
    pages = sum(-(-(c + t) // BLOCK_SIZE) for c, t in seqs) + 8
    rows = 256 if len(seqs) <= 256 else 1024
    eng = Engine(model, EngineConfig(max_num_seqs=rows, max_num_batched_tokens=STEP, max_model_len=max(4096, 1 << (longest - 1).bit_length()),
                                     num_kv_blocks=pages, enable_prefix_caching=False))
    eng.kv.wait_ready()
    eng.alloc.grow(eng.kv.ready_blocks())
    texts, of, fed = _tokens(case, cfg, seed)
    handles = [eng.open_sequence() for _ in seqs]
    # read what stands before the step, a full engine step at a time
    batch, room = [], STEP
    for s, j, (c, _) in zip(handles, of, seqs):
        at = 0
        while at < c:
            n = min(room, c - at)
            batch.append((s, texts[j][at:at + n], []))
            at, room = at + n, room - n
            if room == 0:
                eng.feed(batch)
                batch, room = [], STEP
    if batch:
        eng.feed(batch)
    entries = [(s, t, [len(t) - 1]) for s, t in zip(handles, fed)]
    return {"engine": eng, "entries": entries, "before": [c for c, _ in seqs]}


def run(state):
    logits = state["engine"].feed(state["entries"])
    for (s, _, _), c in zip(state["entries"], state["before"]):
        s.num_cached = c
        del s.prompt[c:]
    return logits


# ---------------------------------------------------------------- exact --

def tolerance(case):
    # The same steps with every product by the library (sums in other orders, norms and rotations apart from the
    # products) differ by 0.007 to 0.023 (most at 6 layers and one sequence), single values by 0.03 to 0.10 of the
    # root mean square: a layer rounds its activations to bf16 several times.
    return {"rel": 0.03, "max": 0.4}


def _rotated(x, pos, theta):
    """Rotation of the halves of every head: x [N, heads, D] in 64 bits at positions pos [N]."""
    D = x.shape[-1]
    f = torch.outer(pos.double(), theta ** (-torch.arange(0, D, 2, device=x.device, dtype=torch.float64) / D))
    c, s = f.cos()[:, None], f.sin()[:, None]
    a, b = x[..., :D // 2], x[..., D // 2:]
    return torch.cat([a * c - b * s, b * c + a * s], -1)


def _attend(q, k, v, first):
    """Causal attention of q [n, Hq, D] at positions first.. over k, v [m, Hkv, D]."""
    n, hq, D = q.shape
    G, out = hq // k.shape[1], torch.empty_like(q)
    for h in range(k.shape[1]):
        kh, vh = k[:, h].t().contiguous(), v[:, h].contiguous()
        for r in range(0, n, 1024):
            m = min(k.shape[0], first + r + 1024)
            qq = q[r:r + 1024, h * G:(h + 1) * G]
            s = (qq.reshape(-1, D) @ kh[:, :m]).view(-1, G, m) / math.sqrt(D)
            at = first + r + torch.arange(qq.shape[0], device=q.device)
            s.masked_fill_(torch.arange(m, device=q.device)[None, None] > at[:, None, None], -math.inf)
            out[r:r + 1024, h * G:(h + 1) * G] = (s.softmax(-1).view(-1, m) @ vh[:m]).view(-1, G, D)
    return out


def _mlp(x, gate, up, down):
    y = torch.empty_like(x)
    for r in range(0, x.shape[0], 4096):
        g = x[r:r + 4096] @ gate.t()
        y[r:r + 4096] = (g * g.sigmoid() * (x[r:r + 4096] @ up.t())) @ down.t()
    return y


def exact(case, seed):
    cfg, seqs = _config(case), _sequences(case)
    texts, of, fed = _tokens(case, cfg, seed)
    D, eps, dev = cfg.head_dim, cfg.rms_eps, "cuda"
    # rows: the texts as far as a sequence has them, then what each sequence is fed
    rows, pos, spans = [], [], []
    for t in texts:
        spans.append((len(rows), len(t)))
        rows, pos = rows + t, pos + list(range(len(t)))
    starts = []
    for (c, t), toks in zip(seqs, fed):
        starts.append(len(rows))
        rows, pos = rows + toks, pos + list(range(c, c + t))
    rows, pos = torch.tensor(rows, device=dev), torch.tensor(pos, device=dev)
    norm = lambda x: x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps)  # noqa: E731
    last = torch.tensor([a + t - 1 for a, (_, t) in zip(starts, seqs)], device=dev)
    for at, w in _weights(cfg, seed):
        if at == "embed":
            h = w[rows].double()
        elif at == "lm_head":
            return norm(h[last]) @ w.double().t()
        else:
            w = {n: t.double() for n, t in w.items()} if not cfg.num_experts else w
            wide = lambda n: w[n].double()  # noqa: E731, B023
            x = norm(h)
            q = _rotated((x @ wide("q").t()).view(-1, cfg.num_heads, D), pos, cfg.rope_theta)
            k = _rotated((x @ wide("k").t()).view(-1, cfg.num_kv_heads, D), pos, cfg.rope_theta)
            v = (x @ wide("v").t()).view(-1, cfg.num_kv_heads, D)
            a = torch.empty_like(q)
            for s, n in spans:
                a[s:s + n] = _attend(q[s:s + n], k[s:s + n], v[s:s + n], 0)
            for s, j, (c, t) in zip(starts, of, seqs):
                p = spans[j][0]
                kk, vv = (torch.cat([y[p:p + c], y[s:s + t]]) for y in (k, v))
                a[s:s + t] = _attend(q[s:s + t], kk, vv, c)
            h = h + a.reshape(len(rows), -1) @ wide("o").t()
            x = norm(h)
            if not cfg.num_experts:
                h = h + _mlp(x, w["gate"], w["up"], w["down"])
                continue
            top, pick = (x @ wide("router").t()).topk(cfg.top_k, dim=-1)
            top = top.softmax(-1)
            for e in range(cfg.num_experts):
                r, slot = (pick == e).nonzero(as_tuple=True)
                y = _mlp(x[r], w["gate"][e].double(), w["up"][e].double(), w["down"][e].double())
                h[r] += y * top[r, slot][:, None]
