"""The work that users of the sampler have it do, as cases that can be timed
and compared: greedy and stochastic sampling of [B, V] logits, decode loops
with histories and stop ids, LM-head logits in the three weight formats, and
one row sampled from host memory.

A case is a dict of plain values:
  kind   "greedy" (argmax_batch), "sample" (sample_batch), "decode" (a burst of
         decode_step calls), "head" (lm_head_logits), "head_greedy"
         (lm_head_greedy), "serve" (lm_head_logits + decode_step, a burst),
         "one" (sample_one: host logits in, token out)
  B, V   rows (sequences) and vocabulary; pad: extra columns per logits row
  T, p, k, pen   temperature, top-p, top-k, repetition penalty
  hist   ids already generated per row (the penalty list); steps: tokens per burst
  dist   what the logits look like: "normal" (sigma), "zipf" (a trained model's
         rank-frequency slope), "peaked" (a few clear favourites over noise),
         "flat" (an uncertain model)
  H, fmt, group  hidden size, weight format (0 f32, 8 int8, 4 int4), scale group
"""
import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "nimbus-infer-rs_amd"))

import nimbus_sampler as ns  # noqa: E402

MASK64 = (1 << 64) - 1


def listed():
    sample = dict(kind="sample", pad=0, k=0, pen=1.0, hist=0, stats=False)
    decode = dict(kind="decode", pad=0)
    return [
        # the smallest call: one interactive sequence, greedy
        dict(name="greedy_one", kind="greedy", B=1, V=50257, pad=0, dist="normal", sigma=3.0),
        # the drop-in call of a host program that keeps its logits in host memory
        dict(name="one_host_row", kind="one", V=50257, T=0.8, p=0.9, k=40, pen=1.1, hist=128,
             dist="normal", sigma=3.0),
        # nucleus sampling of a full batch at a GPT-2 vocabulary: the headline batch
        dict(sample, name="nucleus_batch", B=256, V=50257, T=0.8, p=0.9, dist="normal", sigma=3.0),
        # the largest batch, an uncertain model at a high temperature: nearly every id is kept
        dict(sample, name="nucleus_flat", B=1024, V=50257, T=1.3, p=0.99, dist="flat", sigma=0.0),
        # the largest call: a large batch at a 128k vocabulary
        dict(sample, name="nucleus_long", B=512, V=128256, T=0.8, p=0.9, dist="normal", sigma=2.0),
        # top-k and top-p together at a 128k vocabulary, the ids' probabilities asked for
        dict(sample, name="topk_long_stats", B=64, V=128256, T=0.7, p=0.9, k=50, dist="zipf", sigma=0.0,
             stats=True),
        # a chat server's defaults, every knob on: top-k, top-p and a repetition penalty
        dict(decode, name="decode_all_knobs", B=64, V=50257, T=0.7, p=0.9, k=50, pen=1.1, hist=200,
             steps=8, dist="zipf", sigma=0.0),
        # nucleus sampling with a repetition penalty at a 128k vocabulary
        dict(decode, name="decode_long_penalty", B=128, V=128256, T=0.8, p=0.9, k=0, pen=1.1, hist=256,
             steps=4, dist="normal", sigma=2.0),
        # the tied f32 head of a small model for a full batch
        dict(name="head_f32_batch", kind="head", B=256, H=768, V=50257, fmt=0, group=0),
        # a quantized head of a larger model for a medium batch
        dict(name="head_int8_batch", kind="head", B=64, H=2048, V=128256, fmt=8, group=0),
        # one sequence decoded greedily through a grouped int4 head
        dict(name="head_int4_greedy_one", kind="head_greedy", B=1, H=4096, V=128256, fmt=4, group=128),
        # the whole loop for a ragged batch: head, then sampling with a penalty, a few tokens
        dict(name="serve_ragged", kind="serve", B=17, H=768, V=50257, fmt=8, group=64, T=0.8, p=0.95, k=0,
             pen=1.1, hist=64, steps=4),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _knobs(rng, c, knobs):
    """Sampling knobs as requests carry them; `knobs`: top-k and penalty allowed."""
    c["T"] = round(rng.uniform(0.3, 1.5), 2)
    c["p"] = 1.0 if rng.random() < 0.15 else round(rng.uniform(0.5, 0.99), 2)
    c["k"], c["pen"], c["hist"] = 0, 1.0, 0
    if knobs:
        if rng.random() < 0.6:
            c["k"] = _log_int(rng, 5, 200)
        if c["k"] == 0 or rng.random() < 0.6:
            c["pen"] = round(rng.uniform(1.05, 1.5), 2)
            c["hist"] = _log_int(rng, 8, 1000)
    return c


def _logits_kind(rng, c):
    c["dist"] = rng.choice(["normal", "normal", "zipf", "peaked", "flat"])
    c["sigma"] = round(rng.uniform(1.5, 4.0), 2) if c["dist"] == "normal" else 0.0
    return c


def draw(rng):
    """One more case of the listed ones' ranges."""
    kind = rng.choice(["greedy", "sample", "sample", "sample", "decode", "decode", "head", "head",
                       "head_greedy", "serve", "one"])
    c = dict(kind=kind, V=_log_int(rng, 1000, 262144))
    if kind in ("greedy", "sample", "decode"):
        knobs = kind == "decode" or (kind == "sample" and rng.random() < 0.5)
        most = 16_000_000 if knobs else 65_000_000  # values per call
        c["B"] = _log_int(rng, 1, min(1024, most // c["V"]))
        c["pad"] = rng.choice([0, 0, 1, 3, 64])
        _logits_kind(rng, c)
        if kind != "greedy":
            _knobs(rng, c, knobs)
        if kind == "sample":
            c["stats"] = c["k"] > 0 and rng.random() < 0.5
        if kind == "decode":
            c["steps"] = rng.randint(1, 4)
    elif kind == "one":
        _knobs(rng, _logits_kind(rng, c), True)
    else:
        c["fmt"] = rng.choice([0, 8, 8, 4, 4])
        c["H"] = 8 * _log_int(rng, 32, 512)
        c["group"] = 0
        if c["fmt"] and rng.random() < 0.5:
            c["group"] = rng.choice([g for g in (32, 64, 128) if c["H"] % g == 0] or [0])
        c["V"] = min(c["V"], 67_000_000 // c["H"] if c["fmt"] == 0 else 262_000_000 // c["H"])
        c["B"] = 1
        if kind != "head_greedy":
            c["B"] = _log_int(rng, 1, max(1, min(256, 16_000_000_000 // (c["H"] * c["V"]))))
        if kind == "serve":
            c["steps"] = rng.randint(1, 2)
            c["B"] = min(c["B"], max(1, 8_000_000 // c["V"]))
            _knobs(rng, c, True)
    return c


# ---------------------------------------------------------------------------
# What a user's program has in hand before the call

_sampler = None


def sampler():
    """One sampler context for the whole program."""
    global _sampler
    if _sampler is None:
        _sampler = ns.Sampler(torch.cuda.current_device())
    return _sampler


def _logits(case, B, gen):
    V, pad, dev = case["V"], case.get("pad", 0), "cuda"
    dist = case["dist"]
    x = torch.empty(B, V + pad, dtype=torch.float32, device=dev)
    body = x[:, :V]
    if dist == "normal":
        x.normal_(0.0, case["sigma"], generator=gen)
    elif dist == "flat":
        x.uniform_(-0.5, 0.5, generator=gen)
    elif dist == "peaked":
        x.normal_(0.0, 1.0, generator=gen)
        at = torch.randint(0, V, (B, 4), device=dev, generator=gen)
        up = torch.rand(B, 4, device=dev, generator=gen) * 7.0 + 8.0
        body.scatter_add_(1, at, up)
    else:  # zipf: log-probabilities -1.1 ln(rank) with noise, ranks in a row's own order
        rank = torch.rand(B, V, device=dev, generator=gen).argsort(dim=1).float()
        x.normal_(0.0, 0.5, generator=gen)
        body.sub_(rank.add_(1.0).log_(), alpha=1.1)
    return x


def _history(case, x, gen):
    """Ids that these logits' model would have produced: drawn from their softmax."""
    pr = torch.softmax(x[:, : case["V"]] / case["T"], dim=1)
    return torch.multinomial(pr, case["hist"], replacement=True, generator=gen).to(torch.int32)


def _states(B, seed):
    st = ns.rng_states([seed * 100003 + b for b in range(B)])
    return torch.from_numpy(st.view(np.int64)).cuda()


def _params(case):
    return ns.SamplingParams(temperature=case["T"], top_k=case["k"], top_p=case["p"],
                             repetition_penalty=case["pen"])


def _weights(case, gen):
    """A trained head's weights: f32 rows, or codes with a scale per row or group."""
    V, H, fmt, dev = case["V"], case["H"], case["fmt"], "cuda"
    if fmt == 0:
        return torch.empty(V, H, device=dev).normal_(0.0, 0.05, generator=gen), None
    groups = H // case["group"] if case["group"] else 1
    scales = torch.rand(V, groups, device=dev, generator=gen).add_(0.5).mul_(0.05 / (42.0 if fmt == 8 else 2.4))
    if fmt == 8:  # normal codes, a third of the range per deviation
        codes = torch.empty(V, H, device=dev).normal_(128.0, 42.0, generator=gen).round_().clamp_(0, 255)
        return codes.to(torch.uint8), scales
    n = (V * H + 1) // 2
    lo, hi = (torch.empty(n, device=dev).normal_(8.0, 2.4, generator=gen).round_().clamp_(0, 15)
              .to(torch.uint8) for _ in range(2))
    return lo | (hi << 4), scales


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(int(seed))
    kind, V = case["kind"], case["V"]
    s = dict(case=case, sampler=sampler())
    if kind in ("head", "head_greedy", "serve"):
        B, H = case["B"], case["H"]
        steps = case.get("steps", 1)
        # normalised hidden rows: about unit variance, a few stronger channels
        h = torch.empty(steps, B, H, device="cuda").normal_(0.0, 1.0, generator=gen)
        h[:, :, :: max(1, H // 8)] *= 4.0
        s["hidden"] = h
        s["data"], s["scales"] = _weights(case, gen)
        s["logits"] = torch.empty(B, V, device="cuda")
        s["token"] = torch.zeros(1, dtype=torch.int32, device="cuda")
    if kind == "one":
        x = _logits(case, 1, gen)
        s["generated"] = _history(case, x, gen)[0].tolist() if case["hist"] else []
        s["logits"] = x[0].cpu().numpy()
        s["rng"] = ns.Rng(int(seed))
    if kind in ("greedy", "sample"):
        B = case["B"]
        s["logits"] = _logits(case, B, gen)
        s["tokens"] = torch.zeros(B, dtype=torch.int32, device="cuda")
    if kind == "sample":
        s["rng"] = _states(B, seed)
        s["stats"] = torch.zeros(B, 64, dtype=torch.uint8, device="cuda") if case["stats"] else None
        s["gen_ids"] = s["gen_offsets"] = None
        if case["hist"]:
            s["gen_ids"] = _history(case, s["logits"], gen).reshape(-1)
            s["gen_offsets"] = torch.arange(0, B + 1, dtype=torch.int64, device="cuda") * case["hist"]
    if kind in ("decode", "serve"):
        B, steps, hist = case["B"], case["steps"], case["hist"]
        if kind == "decode":
            s["logits"] = [_logits(case, B, gen) for _ in range(steps)]
        s["rng"] = _states(B, seed)
        s["tokens"] = torch.zeros(steps, B, dtype=torch.int32, device="cuda")
        s["gen_ids"] = torch.zeros(B, hist + steps + 32, dtype=torch.int32, device="cuda")
        if hist and kind == "decode":
            s["gen_ids"][:, :hist] = _history(case, s["logits"][0], gen)
        elif hist:
            s["gen_ids"][:, :hist] = torch.randint(0, V, (B, hist), device="cuda", generator=gen).to(torch.int32)
        s["gen_start"] = torch.full((B,), hist, dtype=torch.int32, device="cuda")
        s["gen_len"] = s["gen_start"].clone()
        s["max_new"] = torch.full((B,), hist + steps + 16, dtype=torch.int32, device="cuda")
        s["done"] = torch.zeros(B, dtype=torch.uint8, device="cuda")
        s["stop"] = torch.tensor([0, V - 1], dtype=torch.int32, device="cuda")
    if kind in ("sample", "decode", "serve", "one"):
        s["params"] = _params(case)
    return s


# ---------------------------------------------------------------------------
# One pass

def _stats(t):
    """The fields of nis_row_stats that the call's contract fixes."""
    f = t.view(torch.float64)
    i = t.view(torch.int32)
    return dict(max_w=f[:, 0], z_kept=f[:, 1], z_all=f[:, 2], u=f[:, 3], prob=f[:, 4],
                kept=t.view(torch.int64)[:, 5], path=i[:, 12], token=i[:, 13])


def run(s):
    case, sm = s["case"], s["sampler"]
    kind, V = case["kind"], case["V"]
    if kind == "greedy":
        return dict(tokens=sm.argmax_batch(s["logits"], V=V, tokens=s["tokens"]))
    if kind == "sample":
        sm.sample_batch(s["logits"], s["params"], s["rng"], V=V, gen_ids=s["gen_ids"],
                        gen_offsets=s["gen_offsets"], tokens=s["tokens"], stats=s["stats"])
        out = dict(tokens=s["tokens"], rng=s["rng"])
        if s["stats"] is not None:
            out["stats"] = _stats(s["stats"])
        return out
    if kind == "one":
        token = sm.sample_one(s["logits"], s["params"], s["generated"], s["rng"])
        return dict(tokens=token, rng=np.array(s["rng"].state(), dtype=np.uint64).view(np.int64))
    if kind == "head":
        return dict(logits=sm.lm_head_logits(s["hidden"][0], case["fmt"], s["data"], V, scales=s["scales"],
                                             group_size=case["group"], out=s["logits"]))
    if kind == "head_greedy":
        token = sm.lm_head_greedy(s["hidden"][0], case["fmt"], s["data"], V, scales=s["scales"],
                                  group_size=case["group"], logits=s["logits"].view(-1), token=s["token"])
        return dict(logits=s["logits"], token=token)
    # a burst of a decode loop: the sequences continue from their histories
    s["gen_len"].copy_(s["gen_start"])
    s["done"].zero_()
    for t in range(case["steps"]):
        if kind == "serve":
            x = sm.lm_head_logits(s["hidden"][t], case["fmt"], s["data"], V, scales=s["scales"],
                                  group_size=case["group"], out=s["logits"])
        else:
            x = s["logits"][t]
        sm.decode_step(x, s["params"], s["rng"], s["gen_ids"], s["gen_len"], s["max_new"], s["done"],
                       stop_ids=s["stop"], V=V, tokens=s["tokens"][t])
    out = dict(tokens=s["tokens"], rng=s["rng"], gen_ids=s["gen_ids"], gen_len=s["gen_len"], done=s["done"])
    if kind == "serve":
        out["logits"] = s["logits"]
    return out


# ---------------------------------------------------------------------------
# What a pass cannot do without, and how exact its results are

def work(case):
    kind, V, steps = case["kind"], case["V"], case.get("steps", 1)
    B = case.get("B", 1)
    nbytes = flops = 0.0
    if kind in ("greedy", "sample", "decode", "one", "serve"):
        per_row = 4 * V + 4 + 4 * case.get("hist", 0)  # logits, token, penalty list
        if kind != "greedy":
            per_row += 64  # RNG state in and out
        if case.get("stats"):
            per_row += 64
        if kind in ("decode", "serve"):
            per_row += 4 + 4 + 1
        nbytes += steps * B * per_row
        flops += steps * B * V * (1 if kind == "greedy" else 2)  # a comparison; a mass and its sum
    if kind in ("head", "head_greedy", "serve"):
        H, fmt = case["H"], case["fmt"]
        weights = V * H * 4 if fmt == 0 else V * H if fmt == 8 else V * H // 2
        if fmt:
            weights += 4 * V * (H // case["group"] if case["group"] else 1)
        nbytes += steps * (weights + 4 * B * H + 4 * B * V)
        flops += steps * 2.0 * B * H * V
    return dict(bytes=nbytes, flops=flops)


def tolerance(case):
    if case["kind"] == "greedy":
        return "exact"
    if case["kind"] in ("head", "head_greedy", "serve"):
        return {"rel": 4e-6, "max": 4e-5, "differ": 0.01}  # f32 sums of up to 4096 products
    return {"rel": 1e-6, "max": 1e-5, "differ": 0.01}  # f32 masses; ids at a boundary of the CDF


def _next_f64(states):
    """xoshiro256++ (Blackman & Vigna) on int64 [B, 4] states: the draws and the next states."""
    s = states.cpu().numpy().view(np.uint64).copy()

    def rotl(x, k):
        return (x << np.uint64(k)) | (x >> np.uint64(64 - k))

    out = rotl(s[:, 0] + s[:, 3], 23) + s[:, 0]
    t = s[:, 1] << np.uint64(17)
    s[:, 2] ^= s[:, 0]
    s[:, 3] ^= s[:, 1]
    s[:, 1] ^= s[:, 2]
    s[:, 0] ^= s[:, 3]
    s[:, 2] ^= t
    s[:, 3] = rotl(s[:, 3], 45)
    u = (out >> np.uint64(11)).astype(np.float64) * 2.0 ** -53
    return torch.from_numpy(u).cuda(), torch.from_numpy(s.view(np.int64)).cuda()


def _sample64(x, case, ids, u):
    """One row each in 64 bits: penalty, temperature, top-k, top-p, inverse CDF in index order.
    x: float64 [n, V] (overwritten); ids: the rows' history lists; u: the rows' draws."""
    pen = float(np.float32(case["pen"]))
    if pen != 1.0 and ids is not None:
        at = ids.long()
        v = x.gather(1, at)
        x.scatter_(1, at, torch.where(v > 0, v / pen, v * pen))
    x /= max(float(np.float32(case["T"])), 1e-6)
    n, V = x.shape
    ninf = float("-inf")
    if 0 < case["k"] < V:
        kth = x.topk(case["k"], dim=1).values[:, -1:]
        x.masked_fill_(x < kth, ninf)
    top = x.max(dim=1, keepdim=True).values
    z_all = torch.zeros(n, dtype=torch.float64, device=x.device)
    p = float(np.float32(case["p"]))
    if p < 1.0:
        order = x.argsort(dim=1, descending=True, stable=True)
        e = torch.exp(x.gather(1, order) - top)
        z_all = e.sum(dim=1)
        e /= z_all[:, None]
        before = e.cumsum(dim=1).sub_(e).sub_(e)  # the running sum before an id, less its own share
        gone = before > p
        x.scatter_(1, order, x.gather(1, order).masked_fill_(gone, ninf))
    m = torch.exp(x - top)
    z = m.sum(dim=1)
    c = m.cumsum(dim=1)
    token = (c >= (u * z)[:, None]).int().argmax(dim=1)
    pr = m.gather(1, token[:, None])[:, 0] / z
    kept = torch.isfinite(x).sum(dim=1)
    return token, dict(max_w=top[:, 0], z_kept=z, z_all=z_all, u=u, prob=pr, kept=kept,
                       path=torch.full_like(token, 4), token=token)


def _head64(h, s, case):
    """Logits of float64 products of the stored weights."""
    V, H, fmt = case["V"], case["H"], case["fmt"]
    out = torch.empty(h.shape[0], V, dtype=torch.float64, device="cuda")
    step = max(2, (1 << 25) // H) & ~1  # an even number of rows keeps int4 rows whole
    for v in range(0, V, step):
        n = min(step, V - v)
        if fmt == 0:
            w = s["data"][v:v + n].double()
        else:
            if fmt == 8:
                q = s["data"][v:v + n].double() - 128.0
            else:
                b = s["data"][v * H // 2:((v + n) * H + 1) // 2]
                q = torch.stack((b & 15, b >> 4), dim=1).reshape(-1)[: n * H].reshape(n, H).double() - 8.0
            g = case["group"] or H
            w = (q.reshape(n, H // g, g) * s["scales"][v:v + n].double()[:, :, None]).reshape(n, H)
        out[:, v:v + n] = h.double() @ w.T
    return out


def exact(case, seed):
    """run()'s floating outputs in 64 bits by plain torch; None for what follows no such value."""
    kind, V = case["kind"], case["V"]
    if kind in ("greedy", "one", "decode"):
        return None
    s = prepare(case, seed)
    if kind == "sample":
        B = case["B"]
        u, rng = _next_f64(s["rng"])
        rows = max(1, 16_000_000 // V)
        token, stats = [], []
        for b in range(0, B, rows):
            n = min(rows, B - b)
            ids = s["gen_ids"].view(B, -1)[b:b + n] if s["gen_ids"] is not None else None
            t, st = _sample64(s["logits"][b:b + n, :V].double(), case, ids, u[b:b + n])
            token.append(t)
            stats.append(st)
        out = dict(tokens=torch.cat(token).int(), rng=rng)
        if case["stats"]:
            st = {f: torch.cat([d[f] for d in stats]) for f in stats[0]}
            out["stats"] = dict(st, path=st["path"].int(), token=st["token"].int())
        return out
    if kind == "head_greedy":
        return dict(logits=_head64(s["hidden"][0], s, case), token=None)
    if kind == "head":
        return dict(logits=_head64(s["hidden"][0], s, case))
    return dict(tokens=None, rng=None, gen_ids=None, gen_len=None, done=None,
                logits=_head64(s["hidden"][-1], s, case))
