"""The sampling work that users of this library give it, as measurable cases.

A case is a dict of plain values. Its "kind" says which public entry point
it goes through:

  step    Sampler.decode_step    one token for B generations whose history
                                 rings, RNG states and done flags live on
                                 the device (a serving loop's inner call)
  sample  Sampler.sample_device  one batch of rows with CSR histories
  head    Sampler.sample_tied_head_device   hidden rows to sampled ids
  host    sample_with            one row in host memory (the CPU sampler's
                                 own signature)

Every output is a whole number or, for the tied head's logits, a binary32
value whose operations and their order are fixed by the reference, so two
correct implementations agree bit for bit.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from scriptonait_amd.sampler import EOS, Rng, Sampler, SamplingConfig, sample_with
from scriptonait_amd.workloads import make_params

# A serving process keeps one context for all of its calls.
_sampler = None


def _handle() -> Sampler:
    global _sampler
    if _sampler is None:
        _sampler = Sampler(0)
    return _sampler


def _step(name, B, V, top_k, window, mask, T=0.9, top_p=0.95, min_p=0.0, rp=1.1, spread=2.0):
    return dict(name=name, kind="step", B=B, V=V, top_k=top_k, window=window, mask=mask, T=T, top_p=top_p,
                min_p=min_p, rp=rp, spread=spread)


def _sample(name, B, V, ld, top_k, H, T, top_p, min_p, rp, spread, hist="uniform", shape="normal"):
    return dict(name=name, kind="sample", B=B, V=V, ld=ld, top_k=top_k, H=H, T=T, top_p=top_p, min_p=min_p, rp=rp,
                spread=spread, hist=hist, shape=shape)


def _head(name, B, V, h):
    return dict(name=name, kind="head", B=B, V=V, h=h, T=0.9, top_k=40, top_p=0.95, min_p=0.0, rp=1.1, H=128)


def listed():
    return [
        # One user's generation with the reference's default parameters and
        # the corpus mask it always passes: a step is launch latency.
        _step("step_one", 1, 8192, 40, 128, "bits", spread=2.0),
        # The drop-in call itself: one row of host logits, default config.
        dict(name="host_one", kind="host", V=32000, H=128, T=0.9, top_k=40, top_p=0.95, min_p=0.0, rp=1.1, spread=2.0,
             masked=True),
        # A small server batch over a small vocabulary, all filters on.
        _step("step_64", 64, 8192, 50, 512, "bits", T=1.0, top_p=0.9, min_p=0.1, rp=1.2, spread=3.0),
        # The headline batch: B=256, V=32000, every filter, a 1024-id history.
        _sample("sample_256", 256, 32000, 32000, 64, 1024, 0.7, 0.95, 0.05, 1.15, 0.0),
        # Long generations: the window holds thousands of earlier draws, many
        # of them among the row's candidates now.
        _step("step_256_long", 256, 32000, 64, 4096, "none", T=0.7, min_p=0.05, rp=1.15, spread=3.0),
        # A wide top-k (near-untruncated sampling with a bound).
        _sample("wide_topk_256", 256, 32000, 32000, 2000, 1024, 0.7, 0.95, 0.05, 1.15, 0.0),
        # A large batch over a 50257-id vocabulary, rows as a framework's
        # matrix product leaves them (an odd stride), default top-k.
        _sample("topk_50257", 1024, 50257, 50257, 50, 128, 1.0, 0.95, 0.0, 1.1, 1.0),
        # A large vocabulary with a wide top-k and a long skewed history.
        _sample("topk1000_131072", 512, 131072, 131072, 1000, 2048, 0.9, 1.0, 0.02, 1.3, 1.0, "zipf", "gumbel"),
        # Nucleus sampling over the whole vocabulary, no top-k.
        _sample("nucleus_50257", 1024, 50257, 50260, 0, 0, 1.0, 0.98, 0.0, 1.0, 1.0),
        # Min-p sampling over a large vocabulary, penalized history.
        _sample("minp_131072", 512, 131072, 131072, 0, 2048, 0.9, 1.0, 0.02, 1.3, 1.0, "zipf", "gumbel"),
        # The tied output head and the sampler in one call: a full batch and
        # one generation.
        _head("head_256", 256, 32000, 512),
        _head("head_1", 1, 32000, 512),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _size(rng, lo, hi, step):
    """A size of the range, half the time a multiple of `step`."""
    n = _log(rng, lo, hi)
    return min(hi, max(step, n // step * step)) if rng.random() < 0.5 else n


def draw(rng):
    kind = rng.choice(("step", "step", "sample", "sample", "wide", "vocab", "head", "host"))
    T, top_p = round(rng.uniform(0.6, 1.1), 2), rng.choice((0.9, 0.95, 0.98, 1.0))
    min_p, rp = rng.choice((0.0, 0.02, 0.05, 0.1)), rng.choice((1.0, 1.1, 1.15, 1.3))
    spread = round(rng.uniform(1.0, 4.0), 1)
    if kind == "step":
        greedy = rng.random() < 0.15
        c = _step("", _log(rng, 1, 512), _size(rng, 4096, 32768, 64), _log(rng, 10, 200), _log(rng, 64, 4096),
                  rng.choice(("bits", "bytes", "none")), 0.0 if greedy else T, top_p, min_p, max(rp, 1.1), spread)
    elif kind == "head":
        while True:
            B, V, h = _log(rng, 1, 256), _size(rng, 4096, 32768, 64), _size(rng, 128, 1024, 16)
            if B * V * h <= 256 * 32000 * 512:
                break
        c = _head("", B, V, h)
    elif kind == "host":
        c = dict(kind="host", V=_size(rng, 4096, 131072, 64), H=_log(rng, 32, 1024), T=T, top_k=_log(rng, 10, 200),
                 top_p=top_p, min_p=min_p, rp=rp, spread=spread, masked=rng.random() < 0.7)
    else:
        while True:
            B, V = _log(rng, 1, 1024), _size(rng, 4096, 131072, 64)
            if B * V <= 1024 * 50257:
                break
        ld = (V + 3) // 4 * 4 if rng.random() < 0.5 else V
        k = 0 if kind == "vocab" else _log(rng, 10, 100) if kind == "sample" else _log(rng, 100, min(4000, V // 2))
        if kind == "vocab" and top_p == 1.0 and min_p == 0.0 and rng.random() < 0.5:
            top_p = 0.95
        c = _sample("", B, V, ld, k, _log(rng, 32, 2048), T, top_p, min_p, rp, spread, rng.choice(("uniform", "zipf")),
                    rng.choice(("normal", "normal", "gumbel")))
    c.pop("name", None)
    return c


def _logits(gen, B, ld, spread, shape="normal"):
    if shape == "gumbel":
        # A heavier upper tail: few candidates stand out.
        return torch.empty(B, ld, device="cuda").exponential_(generator=gen).log_().neg_().mul_(spread)
    x = torch.randn(B, ld, generator=gen, device="cuda")
    if spread == 0.0:
        # Flat rows and peaked rows in turn, as a batch of different prompts has.
        x[0::2] *= 0.5
        x[1::2] *= 4.0
    else:
        x *= spread
    return x


def _history(gen, n, V, how):
    """n token ids: uniform, or Zipf(1) ranks over a seeded permutation."""
    if how == "uniform":
        return torch.randint(0, V, (n,), generator=gen, device="cuda", dtype=torch.int32)
    cdf = torch.cumsum(1.0 / torch.arange(1, V + 1, device="cuda", dtype=torch.float64), 0)
    u = torch.rand(n, generator=gen, device="cuda", dtype=torch.float64) * cdf[-1]
    perm = torch.randperm(V, generator=gen, device="cuda").to(torch.int32)
    return perm[torch.searchsorted(cdf, u).clamp_(max=V - 1)]


def _seen(gen, V):
    """A corpus mask: about nine ids in ten occur in the corpus."""
    return torch.rand(V, generator=gen, device="cuda") < 0.9


def _rng_states(gen, B):
    return torch.randint(-(2 ** 63), 2 ** 63 - 1, (B,), generator=gen, device="cuda", dtype=torch.int64)


def prepare(case, seed):
    c = case
    gen = torch.Generator(device="cuda")
    gen.manual_seed(int(seed))
    if c["kind"] == "host":
        V = c["V"]
        x = _logits(gen, 1, V, c["spread"])[0].cpu().numpy()
        recent = _history(gen, c["H"], V, "zipf").cpu().numpy().astype(np.uint32)
        allowed = _seen(gen, V).cpu().numpy() if c["masked"] else None
        cfg = SamplingConfig(temperature=c["T"], top_k=c["top_k"], top_p=c["top_p"], min_p=c["min_p"],
                             repetition_penalty=c["rp"], repetition_window=c["H"], allowed=allowed)
        return {"kind": "host", "logits": x, "cfg": cfg, "recent": recent, "rng": Rng.seed_from_u64(int(seed) * 7919 + 1)}
    B, V = c["B"], c["V"]
    s = {"kind": c["kind"], "sampler": _handle(), "params": make_params(c["T"], c["top_k"], c["top_p"], c["min_p"], c["rp"]),
         "rng": _rng_states(gen, B), "ids": torch.zeros(B, dtype=torch.int32, device="cuda")}
    if c["kind"] == "step":
        # The model's logits change from step to step: a few sets, taken in turn.
        sets = [_logits(gen, B, V, c["spread"]) for _ in range(4)]
        for x in sets:
            x[:, EOS] = -40.0  # generations that do not end yet
        W = c["window"]
        cap = W + 64
        ring = _history(gen, B * cap, V, "zipf").view(B, cap)
        # A third of the window: earlier draws, that is ids near the top of
        # the row's distributions.
        own = max(1, W // 3)
        top = torch.topk(sets[0], 256, dim=1).indices.to(torch.int32)
        pick = (torch.rand(B, own, generator=gen, device="cuda").square_() * 256).long()
        where = torch.randperm(cap, generator=gen, device="cuda")[:own]
        ring[:, where] = torch.gather(top, 1, pick)
        ring[ring == EOS] = EOS + 1
        s.update(sets=sets, at=0, window=W, ring=ring.contiguous(),
                 ring_len=torch.full((B,), cap, dtype=torch.int32, device="cuda"),
                 done=torch.zeros(B, dtype=torch.int32, device="cuda"), bytes=None, bits=None, V=V)
        if c["mask"] != "none":
            seen = _seen(gen, V)
            if c["mask"] == "bytes":
                s["bytes"] = seen.to(torch.uint8)
            else:
                tokens = torch.nonzero(seen).view(-1).to(torch.int32)
                s["bits"] = s["sampler"].seen_tokens(tokens, V)
        return s
    H = c["H"]
    s["hist"] = s["offs"] = None
    if H:
        s["hist"] = _history(gen, B * H, V, c.get("hist", "zipf"))
        s["offs"] = (torch.arange(B + 1, device="cuda", dtype=torch.int64) * H).to(torch.int32)
    if c["kind"] == "sample":
        s["logits"] = _logits(gen, B, c["ld"], c["spread"], c["shape"])
        s["kept"] = torch.zeros(B, dtype=torch.int32, device="cuda")
        s["V"] = V
    else:
        s["hidden"], s["embed"] = _head_inputs(gen, c)
        s["logits"] = torch.empty(B, V, device="cuda")
    return s


def _head_inputs(gen, c):
    # A normed hidden row has unit mean square; the table is scaled so that
    # logits spread over a few units.
    hidden = torch.randn(c["B"], c["h"], generator=gen, device="cuda")
    embed = torch.randn(c["V"], c["h"], generator=gen, device="cuda") * (2.0 / math.sqrt(c["h"]))
    return hidden, embed


def run(state):
    s = state
    if s["kind"] == "host":
        token = sample_with(s["logits"], s["cfg"], s["recent"], s["rng"])
        return {"id": token, "rng": np.array([s["rng"].state], dtype=np.uint64)}
    if s["kind"] == "step":
        at, s["at"] = s["at"], (s["at"] + 1) % len(s["sets"])
        s["sampler"].decode_step(s["sets"][at], s["params"], s["ring"], s["ring_len"], s["done"], s["window"], s["rng"],
                                 s["ids"], allowed=s["bytes"], allowed_bits=s["bits"], allowed_len=s["V"])
        return {"ids": s["ids"], "rng": s["rng"], "ring": s["ring"], "ring_len": s["ring_len"], "done": s["done"]}
    if s["kind"] == "sample":
        s["sampler"].sample_device(s["logits"], s["params"], s["rng"], s["ids"], V=s["V"], hist=s["hist"],
                                   hist_offsets=s["offs"], out_kept=s["kept"])
        return {"ids": s["ids"], "rng": s["rng"], "kept": s["kept"]}
    s["sampler"].sample_tied_head_device(s["hidden"], s["embed"], s["params"], s["rng"], s["ids"], hist=s["hist"],
                                         hist_offsets=s["offs"], out_logits=s["logits"])
    return {"ids": s["ids"], "rng": s["rng"], "logits": s["logits"]}


def work(case):
    c = case
    V, B = c["V"], c.get("B", 1)
    # RNG state in and out, the id out, the row's history ids.
    per_row = 8 + 8 + 4 + (4 * c.get("H", c.get("window", 0)) if c["rp"] != 1.0 and c["kind"] != "head" else 0)
    mask = V // 8 if c.get("mask") == "bits" else V if c.get("mask") == "bytes" or c.get("masked") else 0
    if c["kind"] == "head":
        h = c["h"]
        return {"bytes": 4 * (V * h + B * h + B * V) + B * (per_row + 4 * c["H"]), "flops": 2 * B * V * h}
    return {"bytes": B * (4 * V + per_row) + mask, "flops": 0}


def tolerance(case):
    # Ids, counts and states are whole numbers, and the head's logits follow
    # the reference's dot product operation by operation.
    return "exact"


def exact(case, seed):
    if case["kind"] != "head":
        return None
    c = case
    gen = torch.Generator(device="cuda")
    gen.manual_seed(int(seed))
    _rng_states(gen, c["B"])
    if c["H"]:
        _history(gen, c["B"] * c["H"], c["V"], "zipf")
    hidden, embed = _head_inputs(gen, c)
    return {"ids": None, "rng": None, "logits": hidden.double() @ embed.double().t()}
