"""The work whose speed is measured: what a program of this framework has its
engine do, through the public calls of ana_amd.Decoder.

A case is a dict of plain values:

- kind: "turn" (one token fed into each sequence, then the logits: a program
  that picks on the host), "greedy" and "sampled" (the token loop on the
  device, then the logits), "prompt" (slots emptied, prompts fed, the logits
  of their last tokens), "score" (slots emptied, windows scored).
- model: "115m" (d 768, MLP 2048, 12 layers, 12 heads, vocabulary 32768,
  context 2048, RG-LRU, qk-norm and sinks on), "v2" (the same widths at
  context 256, the three off) or "v1" (d 256, MLP 1024, 4 layers, 4 heads,
  context 256, the three off).
- mode: "exact", "fast_fp32" or "bf16".
- n: sequences; length: the longest prompt or window, in tokens; spread: the
  sequences' lengths go down evenly from length to length - spread; steps:
  tokens a loop decodes; chunk: the Decoder's prefill_chunk; emb: the
  embedding's standard deviation.

A case's checkpoint is random (gains, qk gains and sinks as a trained model
has them, residual products scaled down with depth) and the same for every
seed, as a program's is; the seed makes the prompts. With emb 0.04 the
residual stream keeps enough of a token for greedy picks to have the margins
that a trained model's have (rounding does not decide them); the sampled
cases take 0.02, whose distributions are flat enough to be drawn from.
"""
import hashlib
import math
import os
import tempfile

import numpy as np
import torch

import ana_amd
from ana_amd import ckpt
from ana_amd import config as cf

MODELS = {"115m": cf.FP100M, "v2": cf.V2, "v1": cf.V1}
MODES = {"exact": ana_amd.EXACT_FP32, "fast_fp32": ana_amd.FAST_FP32, "bf16": ana_amd.BF16}
WIDE, FLAT = 0.04, 0.02
TEMPERATURE, TOP_K, TOP_P = float(np.float32(0.8)), 40, float(np.float32(0.9))


def _case(name, kind, model, mode, n, length, spread=0, steps=0, chunk=64, emb=WIDE):
    c = {"kind": kind, "model": model, "mode": mode, "n": n, "length": length, "spread": spread, "steps": steps,
         "chunk": chunk, "emb": emb}
    return dict(c, name=name) if name else c


def listed():
    return [
        # the smallest call: one token into the smallest model in the default
        # mode, its logits read back (a host that picks by itself)
        _case("turn_v1_1_exact", "turn", "v1", "exact", 1, 33),
        # one user's stream deep in a full window, in each mode
        _case("greedy_1_fast", "greedy", "115m", "fast_fp32", 1, 1920, steps=32),
        _case("greedy_1_bf16", "greedy", "115m", "bf16", 1, 301, steps=32),
        _case("greedy_1_exact", "greedy", "115m", "exact", 1, 500, steps=16),
        # a full batch: short prompts, then ragged ones
        _case("greedy_64_fast", "greedy", "115m", "fast_fp32", 64, 128, steps=32),
        _case("greedy_64_bf16", "greedy", "115m", "bf16", 64, 512, spread=400, steps=32),
        # long conversations: half a batch with the whole window live
        _case("greedy_32_deep_fast", "greedy", "115m", "fast_fp32", 32, 1920, spread=101, steps=16, chunk=128),
        # sampled chat traffic (temperature, top-k and top-p all on)
        _case("sampled_64_fast", "sampled", "115m", "fast_fp32", 64, 128, steps=16, chunk=128, emb=FLAT),
        # a batch of prompts coming in, in both fast modes
        _case("prompt_64_bf16", "prompt", "115m", "bf16", 64, 512, chunk=128),
        _case("prompt_64_fast", "prompt", "115m", "fast_fp32", 64, 512, chunk=128),
        # one long prompt at the default chunk: the time to its first token
        _case("prompt_1_fast", "prompt", "115m", "fast_fp32", 1, 1919),
        # the evaluator's windows in the default mode
        _case("score_8_exact", "score", "115m", "exact", 8, 257),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["turn", "greedy", "greedy", "sampled", "prompt", "prompt", "score"])
    mode = rng.choice(["exact", "fast_fp32", "fast_fp32", "bf16"])
    model = rng.choice(["115m", "115m", "115m", "v2", "v1"])
    ctx = MODELS[model].ctx
    chunk = rng.choice([64, 64, 128])
    emb = FLAT if kind == "sampled" else WIDE
    # the most tokens a pass (or its preparation) feeds: the exact mode's
    # products take many times as long
    most = 1500 if mode == "exact" else 32768
    if kind in ("prompt", "score"):
        n = _log(rng, 1, 16 if mode == "exact" else 64)
        length = min(_log(rng, 9, ctx), max(9, most // n))
        return _case("", kind, model, mode, n, length, rng.randrange(0, length // 2), chunk=chunk, emb=emb)
    n = _log(rng, 1, 64)
    # (draws sit on the edges of a distribution that bf16 rounding moves)
    if kind == "sampled" and mode == "bf16":
        mode = "fast_fp32"
    steps = 0 if kind == "turn" else _log(rng, 2, 16)
    length = min(_log(rng, 9, ctx - 20), max(9, 2 * most // n))
    return _case("", kind, model, mode, n, length, rng.randrange(0, length // 2), steps, chunk, emb)


# ---------------------------------------------------------------- the inputs

def _device():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _weights(case):
    """The checkpoint's parameters as (name, tensor) in the file's order."""
    c, dev = MODELS[case["model"]], _device()
    g = torch.Generator(device=dev)
    g.manual_seed(20240)
    d, f = c.d, c.f

    def normal(shape, std, base=0.0):
        return torch.randn(shape, generator=g, device=dev, dtype=torch.float32) * std + base

    out = [("emb", normal((c.vocab, d), case["emb"]))]
    deep = 0.02 / math.sqrt(2 * c.layers)
    for i in range(c.layers):
        b = [("ra", normal(d, 0.1, 1.0)), ("wq", normal((d, d), 0.02)), ("wk", normal((d, d), 0.02)),
             ("wv", normal((d, d), 0.02)), ("wo", normal((d, d), deep))]
        if not c.is_softmax(i):
            b.append(("wa", normal((d, d), 0.02)))
            if c.rglru:
                # sigmoid(lam)^8 uniform on [0.9, 0.999)
                u = torch.rand(d, generator=g, device=dev, dtype=torch.float64) * 0.099 + 0.9
                a = u ** 0.125
                b.append(("lam", torch.log(a / (1 - a)).float()))
        else:
            if c.qk:
                b += [("gq", normal(c.hd, 0.1)), ("gk", normal(c.hd, 0.1))]
            if c.sinks:
                b.append(("sink", normal(c.heads, 1.0)))
        b += [("rf", normal(d, 0.1, 1.0)), ("wg", normal((f, d), 0.02)), ("wu", normal((f, d), 0.02)),
              ("wd", normal((d, f), deep))]
        out += [(f"{i}.{k}", t) for k, t in b]
    return out + [("final", normal(d, 0.1, 1.0))]


def _checkpoint(case):
    """The case's checkpoint file, written once a machine."""
    c = MODELS[case["model"]]
    key = hashlib.sha256(f"1 {c.show()} {case['emb']}".encode()).hexdigest()[:16]
    path = os.path.join(tempfile.gettempdir(), f"ana_cases_{os.getuid()}_{key}.ftc2")
    if not os.path.exists(path):
        flat = torch.cat([t.reshape(-1) for _, t in _weights(case)])
        if flat.numel() != c.params:
            raise ValueError(f"{flat.numel()} parameters, the config has {c.params}")
        big = flat.view(torch.uint8).reshape(-1, 4).flip(1).contiguous().cpu().numpy()
        count = np.array([c.params], dtype=">u8").tobytes()
        tmp = f"{path}.{os.getpid()}"
        with open(tmp, "wb") as fp:
            fp.write(ckpt.manifest_bytes(c) + count)
            big.tofile(fp)
            fp.write(bytes(8) + count)
        os.replace(tmp, path)
    return path


def _lengths(case):
    """Every sequence's prompt or window length."""
    n = case["n"]
    return [max(2, case["length"] - case["spread"] * i // n) for i in range(n)]


def _tokens(case, seed):
    """Each sequence's ids: BOS, then uniform ones."""
    r = np.random.RandomState(seed % (1 << 32))
    v = MODELS[case["model"]].vocab
    return [np.concatenate([[0], r.randint(2, v, k - 1)]).astype(np.uint32) for k in _lengths(case)]


def prepare(case, seed):
    n = case["n"]
    toks = _tokens(case, seed)
    dec = ana_amd.Decoder(_checkpoint(case), max_seqs=n, prefill_chunk=case["chunk"], numerics=MODES[case["mode"]])
    s = {"case": case, "dec": dec, "seqs": list(range(n)), "zero": [0] * n, "toks": toks}
    if case["kind"] in ("turn", "greedy", "sampled"):
        # the conversation so far, all but the token that comes next
        dec.feeds_n(s["seqs"], s["zero"], [t[:-1] for t in toks])
        s["pos"] = [t.size - 1 for t in toks]
        s["next"] = [int(t[-1]) for t in toks]
    if case["kind"] == "sampled":
        s["settings"] = ana_amd.Settings(TEMPERATURE, TOP_K, TOP_P)
        s["rng"] = np.ascontiguousarray(np.stack([ana_amd.rng_seeded(seed + b) for b in range(n)]))
    return s


def run(s):
    dec, seqs, case = s["dec"], s["seqs"], s["case"]
    kind = case["kind"]
    if kind == "turn":
        dec.feed(seqs, s["pos"], s["next"])
        return {"logits": dec.logits(seqs)}
    if kind == "greedy":
        picks = dec.generate(seqs, s["pos"], s["next"], case["steps"])
        return {"picks": picks.astype(np.int64), "logits": dec.logits(seqs)}
    if kind == "sampled":
        rng = s["rng"].copy()
        picks = dec.generate(seqs, s["pos"], s["next"], case["steps"], s["settings"], rng)
        return {"picks": picks.astype(np.int64), "rng": rng.view(np.int64), "logits": dec.logits(seqs)}
    for q in seqs:
        dec.reset(q)
    if kind == "prompt":
        dec.feeds_n(seqs, s["zero"], s["toks"])
        return {"logits": dec.logits(seqs)}
    return {"loss": np.concatenate(dec.score_n(seqs, s["zero"], s["toks"]))}


# ---------------------------------------------------------------- what a pass cannot do without

def work(case):
    c = MODELS[case["model"]]
    wb = 2.0 if case["mode"] == "bf16" else 4.0
    layer_w, head_w = float(c.params - c.vocab * c.d), float(c.vocab * c.d)
    lens, kind, n = _lengths(case), case["kind"], case["n"]
    gla = c.gla_layers * 2.0 * c.heads * c.hd * c.hd * 4.0      # a sequence's states, read and written
    row = 2.0 * c.d * 4.0                                       # a token's k and v in one softmax layer
    by = fl = 0.0
    if kind in ("turn", "greedy", "sampled"):
        steps = max(1, case["steps"])
        for k in range(steps):
            by += wb * (layer_w + head_w)
            fl += 2.0 * n * (layer_w + head_w)
            for t in lens:
                live = min(t + k, c.ctx)
                by += gla + c.softmax_layers * row * (live + 1)
                fl += c.softmax_layers * 4.0 * live * c.d + c.gla_layers * 4.0 * c.heads * c.hd * c.hd
        by += 4.0 * n * c.vocab + (wb * head_w if steps > 1 else 0.0)
        fl += 2.0 * n * head_w if steps > 1 else 0.0
        return {"bytes": by, "flops": fl}
    fed = [t - (kind == "score") for t in lens]
    total = float(sum(fed))
    by = wb * (layer_w + head_w) + n * gla / 2 + c.softmax_layers * row * total
    fl = 2.0 * layer_w * total + total * c.gla_layers * 4.0 * c.heads * c.hd * c.hd
    fl += sum(c.softmax_layers * 2.0 * t * t * c.d for t in fed)
    if kind == "prompt":
        return {"bytes": by + 4.0 * n * c.vocab, "flops": fl + 2.0 * n * head_w}
    return {"bytes": by + 4.0 * total, "flops": fl + 2.0 * total * head_w}


def tolerance(case):
    # exact_fp32 is held to the bit; the others as measured against sums in
    # another order (bf16 rounds every product's activations once)
    if case["mode"] == "exact":
        return "exact"
    if case["mode"] == "bf16":
        return {"rel": 2e-2, "max": 0.2, "differ": 0.01}
    return {"rel": 4e-5, "max": 1e-3, "differ": 0.005}


# ---------------------------------------------------------------- in 64 bits

def _norm(x, g):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + 1e-5) * g


class _Model:
    """The decoder in 64 bits: every sequence's states, any number of tokens
    at once."""

    def __init__(self, case, slots):
        self.c = c = MODELS[case["model"]]
        self.w = {k: t.double() for k, t in _weights(case)}
        self.dev = self.w["emb"].device
        n = case["n"]
        z = lambda *s: torch.zeros(s, dtype=torch.float64, device=self.dev)  # noqa: E731
        self.S = {i: z(n, c.heads, c.hd, c.hd) for i in range(c.layers) if not c.is_softmax(i)}
        self.kv = {i: (z(n, c.heads, slots, c.hd), z(n, c.heads, slots, c.hd))
                   for i in range(c.layers) if c.is_softmax(i)}

    def _gla(self, i, y, live):
        c, w = self.c, self.w
        n, T, _ = y.shape
        heads = lambda t: t.view(n, T, c.heads, c.hd)  # noqa: E731
        q, k, v, z = (heads(y @ w[f"{i}.{m}"].T) for m in ("wq", "wk", "wv", "wa"))
        q, k = (t / torch.sqrt((t * t).sum(-1, keepdim=True) + 1e-6) for t in (q, k))
        if c.rglru:
            cap = -float(np.float32(1e-4))
            lam = torch.nn.functional.logsigmoid(w[f"{i}.lam"]).view(c.heads, c.hd)
            la = torch.clamp(8.0 * torch.sigmoid(z) * lam, max=cap)
            k, al = k * torch.sqrt(-torch.expm1(2.0 * la)), torch.exp(la)
        else:
            al = torch.sigmoid(z)
        on = live.view(n, T, 1, 1)
        al, k = torch.where(on, al, 1.0), torch.where(on, k, 0.0)
        S, o = self.S[i], torch.empty_like(v)
        for t in range(T):
            S.mul_(al[:, t].unsqueeze(-1)).add_(k[:, t].unsqueeze(-1) * v[:, t].unsqueeze(-2))
            o[:, t] = (q[:, t].unsqueeze(-2) @ S).squeeze(-2)
        return o.reshape(n, T, c.d)

    def _attention(self, i, y, pos):
        c, w = self.c, self.w
        n, T, _ = y.shape
        q, k, v = (((y @ w[f"{i}.{m}"].T).view(n, T, c.heads, c.hd)) for m in ("wq", "wk", "wv"))
        if c.qk:
            q, k = _norm(q, 1.0 + w[f"{i}.gq"]), _norm(k, 1.0 + w[f"{i}.gk"])
        K, V = self.kv[i]
        o = torch.empty_like(q)
        sink = w[f"{i}.sink"].view(-1, 1, 1) if c.sinks else torch.full((c.heads, 1, 1), -math.inf, device=self.dev,
                                                                       dtype=torch.float64)
        for b in range(n):
            p = pos[b]
            K[b][:, p], V[b][:, p] = k[b].transpose(0, 1), v[b].transpose(0, 1)
            top = int(p[-1]) + 1
            s = (q[b].transpose(0, 1) @ K[b][:, :top].transpose(1, 2)) / math.sqrt(c.hd)
            at = torch.arange(top, device=self.dev)
            s = s.masked_fill((at > p[:, None]) | (at <= p[:, None] - c.ctx), -math.inf)
            s = torch.softmax(torch.cat([s, sink.expand(-1, T, 1)], -1), -1)[..., :top]
            o[b] = (s @ V[b][:, :top]).transpose(0, 1)
        return o.reshape(n, T, c.d)

    def feed(self, toks, pos0, live):
        """toks, live: [n, T] (a row's tokens past its end count for nothing);
        returns the residual rows [n, T, d]."""
        c, w = self.c, self.w
        x = w["emb"][toks]
        pos = pos0[:, None] + torch.arange(toks.shape[1], device=self.dev)
        for i in range(c.layers):
            y = _norm(x, w[f"{i}.ra"])
            x = x + (self._attention(i, y, pos) if c.is_softmax(i) else self._gla(i, y, live)) @ w[f"{i}.wo"].T
            y = _norm(x, w[f"{i}.rf"])
            x = x + (torch.nn.functional.silu(y @ w[f"{i}.wg"].T) * (y @ w[f"{i}.wu"].T)) @ w[f"{i}.wd"].T
        return x

    def prompts(self, toks):
        """Whole prompts from position 0; the residual rows [n, longest, d]."""
        T = max(t.size for t in toks)
        ids = np.zeros((len(toks), T), dtype=np.int64)
        live = np.zeros((len(toks), T), dtype=bool)
        for b, t in enumerate(toks):
            ids[b, :t.size], live[b, :t.size] = t, True
        return self.feed(torch.from_numpy(ids).to(self.dev), torch.zeros(len(toks), dtype=torch.int64, device=self.dev),
                         torch.from_numpy(live).to(self.dev))

    def logits(self, x):
        return _norm(x, self.w["final"]) @ self.w["emb"].T


def _next_word(r):
    """The xoshiro draw of a row's four words."""
    m = (1 << 64) - 1
    rot = lambda v, k: ((v << k) | (v >> (64 - k))) & m  # noqa: E731
    s0, s1, s2, s3 = r
    word = rot(s1 * 5 & m, 7) * 9 & m
    r[:] = [s0 ^ s3 ^ s1 ^ s2, s1 ^ s2, s2 ^ s0 ^ (s1 << 17 & m), rot(s3 ^ s1, 45)]
    return word


def _seeded(seed):
    m, r = (1 << 64) - 1, []
    for _ in range(4):
        seed = seed + 0x9E3779B97F4A7C15 & m
        z = (seed ^ seed >> 30) * 0xBF58476D1CE4E5B9 & m
        z = (z ^ z >> 27) * 0x94D049BB133111EB & m
        r.append(z ^ z >> 31)
    return r


def _sample(lg, words):
    """Temperature, top-k, top-p and one inverse-CDF draw a row."""
    kept = lg >= torch.topk(lg, TOP_K).values[:, -1:]
    w = torch.where(kept, torch.exp((lg - lg.max(-1, keepdim=True).values) / TEMPERATURE), 0.0)
    top, _ = torch.sort(w, descending=True)
    last = (torch.cumsum(top, -1) < TOP_P * w.sum(-1, keepdim=True)).sum(-1, keepdim=True)
    w = torch.where(w >= torch.gather(top, 1, last), w, 0.0)
    u = torch.tensor([(_next_word(r) >> 40) / 16777216.0 for r in words], dtype=torch.float64, device=lg.device)
    return (torch.cumsum(w, -1) <= (u * w.sum(-1))[:, None]).sum(-1).clamp(max=lg.shape[1] - 1)


def exact(case, seed):
    toks, kind, n = _tokens(case, seed), case["kind"], case["n"]
    with torch.no_grad():
        m = _Model(case, max(t.size for t in toks) + case["steps"])
        rows = torch.arange(n, device=m.dev)
        ends = torch.tensor([t.size for t in toks], device=m.dev) - 1
        if kind == "prompt":
            return {"logits": m.logits(m.prompts(toks)[rows, ends]).cpu().numpy()}
        if kind == "score":
            x = m.prompts([t[:-1] for t in toks])
            out = []
            for b, t in enumerate(toks):
                lg = m.logits(x[b, :t.size - 1])
                want = torch.from_numpy(t[1:].astype(np.int64)).to(m.dev)
                out.append(torch.logsumexp(lg, -1) - lg[torch.arange(t.size - 1, device=m.dev), want])
            return {"loss": torch.cat(out).cpu().numpy()}
        m.prompts([t[:-1] for t in toks])
        on = torch.ones((n, 1), dtype=torch.bool, device=m.dev)
        tok, pos, picks = torch.tensor([int(t[-1]) for t in toks], device=m.dev), ends.clone(), []
        words = [_seeded(seed + b) for b in range(n)]
        for _ in range(max(1, case["steps"])):
            lg = m.logits(m.feed(tok[:, None], pos, on)[:, 0])
            tok = _sample(lg, words) if kind == "sampled" else lg.argmax(-1)
            pos = pos + 1
            picks.append(tok)
        if kind == "turn":
            return {"logits": lg.cpu().numpy()}
        out = {"picks": torch.stack(picks, 1).cpu().numpy(), "logits": lg.cpu().numpy()}
        if kind == "sampled":
            out["rng"] = np.array([[w - (1 << 64) if w >> 63 else w for w in r] for r in words], dtype=np.int64)
        return out
