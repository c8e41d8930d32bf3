"""The attention calls whose speed this repository is measured by.

Each case is one call of the public API as a program makes it: a prefill or encoder
forward, a training step's forward and backward through autograd, a packed
(variable-length) batch in either direction, or one decode step against a KV cache.
`listed()` holds fixed cases, `draw(rng)` samples the ranges they stand for.  The file is
imported with the repository's root as the working folder.
"""

import math
import os
import sys

import torch

_PKG = os.path.join(os.getcwd(), "flash-attention-legacy_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

from flash_attn_legacy import flash_attention, flash_attn_varlen_func, flash_attn_with_kvcache  # noqa: E402

# Upper ends of what a drawn case may cost; both lie below the largest listed cases.
_MAX_FLOPS = 4.0e11
_MAX_BYTES = 1.5e9


def listed():
    return [
        # One user's chat step: a single new token against a half-filled cache in the
        # head-major layout that Hugging Face caches use.  Launches and latency count.
        dict(name="decode_token", kind="decode", batch=1, heads_q=32, heads_kv=8, dim=128, dtype="bfloat16",
             layout="bhsd", capacity=2048, min_len=1000, max_len=1000),
        # A serving step: 32 users with contexts of 1k to 32k tokens (the benchmark's decode
        # configuration).  Bound by reading the cache.
        dict(name="decode_batch", kind="decode", batch=32, heads_q=32, heads_kv=8, dim=128, dtype="float16",
             layout="bshd", capacity=32768, min_len=1024, max_len=32768),
        # A short prompt batch of a small model (the benchmark's small forward): fewer
        # workgroups than compute units.
        dict(name="prefill_small", kind="prefill", batch=2, heads_q=8, heads_kv=8, nq=1024, nk=1024, dim=64,
             dtype="float16", causal=True, layout="bhnd"),
        # One prompt of an odd length through grouped-query heads, as [B, N, H, d]
        # projections seen through a transpose.
        dict(name="prefill_prompt", kind="prefill", batch=1, heads_q=32, heads_kv=8, nq=1531, nk=1531, dim=128,
             dtype="bfloat16", causal=True, layout="bnhd"),
        # A batch of long prompts (the benchmark's headline forward): matrix-core bound.
        dict(name="prefill_large", kind="prefill", batch=4, heads_q=32, heads_kv=8, nq=4096, nk=4096, dim=128,
             dtype="float16", causal=True, layout="bhnd"),
        # An encoder layer over patches: no mask, a ragged length, 12 heads of 64.
        dict(name="encoder", kind="prefill", batch=16, heads_q=12, heads_kv=12, nq=577, nk=577, dim=64,
             dtype="bfloat16", causal=False, layout="bnhd"),
        # A training step's attention layer (the benchmark's backward shape).
        dict(name="train_d128", kind="train", batch=2, heads_q=16, heads_kv=16, nq=2048, nk=2048, dim=128,
             dtype="float16", causal=True, layout="bhnd"),
        # The same with 64-wide heads, in bf16, from transposed projections.
        dict(name="train_d64", kind="train", batch=4, heads_q=16, heads_kv=16, nq=2048, nk=2048, dim=64,
             dtype="bfloat16", causal=True, layout="bnhd"),
        # The widest supported head in training, grouped-query.
        dict(name="train_d256", kind="train", batch=2, heads_q=16, heads_kv=8, nq=2048, nk=2048, dim=256,
             dtype="bfloat16", causal=True, layout="bnhd"),
        # One long sequence packed with short ones (a scenario of the packed-vs-padded
        # benchmark): small enough that launches and the per-tile lookups count.
        dict(name="varlen_small", kind="varlen", seqs=16, min_len=32, max_len=1024, spread="one_long", heads_q=8,
             heads_kv=8, dim=64, dtype="float16", causal=True),
        # Prefill of 16 packed prompts of 64 to 4096 tokens (the benchmark's packed forward).
        dict(name="varlen_prefill", kind="varlen", seqs=16, min_len=64, max_len=4096, spread="uniform", heads_q=32,
             heads_kv=8, dim=128, dtype="float16", causal=True),
        # A training step over 16 packed documents.
        dict(name="varlen_train", kind="varlen_train", seqs=16, min_len=64, max_len=2048, spread="uniform",
             heads_q=32, heads_kv=8, dim=128, dtype="bfloat16", causal=True),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the ranges above: every kind of call, all head dims with 64 and 128
    most often, both element types, lengths over three orders of magnitude."""
    while True:
        kind = rng.choice(["decode", "decode", "prefill", "prefill", "prefill", "train", "train", "train",
                           "varlen", "varlen_train"])
        heads_q, heads_kv = rng.choice([(8, 8), (16, 16), (12, 12), (32, 32), (32, 8), (32, 8), (16, 8), (16, 4), (8, 1),
                                        (28, 4)])
        case = dict(kind=kind, heads_q=heads_q, heads_kv=heads_kv,
                    dim=rng.choice([32, 64, 64, 64, 96, 128, 128, 128, 128, 256]),
                    dtype=rng.choice(["float16", "bfloat16"]))
        if kind == "decode":
            hi = _log_int(rng, 64, 32768)
            case.update(batch=_log_int(rng, 1, 96), layout=rng.choice(["bshd", "bhsd"]), max_len=hi,
                        min_len=rng.choice([hi, max(1, hi // 8)]), capacity=(hi + rng.randrange(1, hi + 1) + 15) // 16 * 16)
            # the whole capacity counts, so that the state stays within the listed one's
            if case["batch"] * case["capacity"] * heads_kv * case["dim"] * 4 > 2 * _MAX_BYTES:
                continue
        elif kind in ("prefill", "train"):
            nq = _log_int(rng, 64, 8192)
            nk = nq if kind == "train" or rng.random() < 0.8 else _log_int(rng, 64, 4096)
            case.update(batch=_log_int(rng, 1, 16), nq=nq, nk=nk, causal=nk == nq and rng.random() < 0.7,
                        layout=rng.choice(["bhnd", "bnhd"]))
        else:
            hi = _log_int(rng, 128, 6144)
            case.update(seqs=_log_int(rng, 2, 100), max_len=hi, min_len=max(1, hi // rng.choice([4, 16, 64])),
                        spread=rng.choice(["uniform", "uniform", "one_long"]), causal=rng.random() < 0.8)
        w = work(case)
        if 2.0e6 < w["flops"] < _MAX_FLOPS and w["bytes"] < _MAX_BYTES:
            return case


def _lengths(case):
    """The segment (or cache) lengths of a case: fixed by its sizes, spread evenly over
    [min_len, max_len] in a scrambled order, the ends included."""
    lo, hi = case["min_len"], case["max_len"]
    n = case["seqs"] if "seqs" in case else case["batch"]
    if case.get("spread") == "one_long":
        return [hi] + [lo] * (n - 1)
    if n == 1:
        return [hi]
    step = next(s for s in (7, 11, 13, 17, 19, 23) if math.gcd(s, n) == 1)
    return [lo + (hi - lo) * (i * step % n) // (n - 1) for i in range(n)]


def _pairs(case):
    """(query, key) pairs per query head, half of them under a causal mask."""
    if case["kind"] in ("prefill", "train"):
        p = float(case["batch"]) * case["nq"] * case["nk"]
    else:
        p = sum(float(n) * n for n in _lengths(case))
    return p / 2 if case["causal"] else p


def work(case):
    hq, hkv, d = case["heads_q"], case["heads_kv"], case["dim"]
    if case["kind"] == "decode":
        rows = float(sum(_lengths(case)))
        return dict(bytes=2.0 * d * (2 * hkv * rows + 2 * hq * case["batch"]), flops=4.0 * hq * d * rows)
    fwd = 4.0 * hq * d * _pairs(case)
    if case["kind"] in ("prefill", "train"):
        tq, tk = float(case["batch"]) * case["nq"], float(case["batch"]) * case["nk"]
    else:
        tq = tk = float(sum(_lengths(case)))
    q, kv = 2.0 * d * hq * tq, 2.0 * d * hkv * tk      # one Q-shaped, one K-shaped tensor
    if case["kind"] in ("prefill", "varlen"):
        return dict(bytes=2 * q + 2 * kv, flops=fwd)
    # q, k, v, dO in; O, dQ, dK, dV out; five products in the backward for two forward
    return dict(bytes=4 * q + 4 * kv, flops=3.5 * fwd)


def _inputs(case, seed):
    """Unit-normal activations, as attention inputs after normalisation layers are."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    dtype = getattr(torch, case["dtype"])
    hq, hkv, d = case["heads_q"], case["heads_kv"], case["dim"]
    rnd = lambda *shape: torch.randn(shape, generator=gen, device="cuda", dtype=dtype)
    if case["kind"] == "decode":
        b, s = case["batch"], case["capacity"]
        cache = (b, s, hkv, d) if case["layout"] == "bshd" else (b, hkv, s, d)
        return dict(q=rnd(b, 1, hq, d), k=rnd(*cache), v=rnd(*cache))
    if case["kind"] in ("prefill", "train"):
        b = case["batch"]
        if case["layout"] == "bnhd":
            heads = lambda h, n: rnd(b, n, h, d).transpose(1, 2)
        else:
            heads = lambda h, n: rnd(b, h, n, d)
        x = dict(q=heads(hq, case["nq"]), k=heads(hkv, case["nk"]), v=heads(hkv, case["nk"]))
        if case["kind"] == "train":
            x["do"] = heads(hq, case["nq"])
        return x
    t = sum(_lengths(case))
    x = dict(q=rnd(t, hq, d), k=rnd(t, hkv, d), v=rnd(t, hkv, d))
    if case["kind"] == "varlen_train":
        x["do"] = rnd(t, hq, d)
    return x


def prepare(case, seed):
    state = dict(case=case, **_inputs(case, seed))
    if case["kind"] == "decode":
        state["lens"] = torch.tensor(_lengths(case), dtype=torch.int32, device="cuda")
    elif case["kind"] in ("varlen", "varlen_train"):
        lens = torch.tensor([0] + _lengths(case))
        state["cu"] = lens.cumsum(0).to(device="cuda", dtype=torch.int32)
        state["max_len"] = int(lens.max())
    if case["kind"] in ("train", "varlen_train"):
        for name in ("q", "k", "v"):
            state[name].requires_grad_(True)
    return state


def run(state):
    case = state["case"]
    q, k, v = state["q"], state["k"], state["v"]
    if case["kind"] == "decode":
        return flash_attn_with_kvcache(q, k, v, state["lens"], cache_layout=case["layout"])
    if case["kind"] in ("prefill", "train"):
        o = flash_attention(q, k, v, is_causal=case["causal"])
    else:
        o = flash_attn_varlen_func(q, k, v, state["cu"], state["cu"], state["max_len"], state["max_len"],
                                   causal=case["causal"])
    if "do" not in state:
        return o
    return (o.detach(), *torch.autograd.grad(o, (q, k, v), state["do"]))


def tolerance(case):
    """Relative 2-norm error and largest error over the root mean square (or the value):
    about four times the error measured against 64 bits over the listed cases and 24 drawn
    ones, which the 16-bit outputs, probabilities and score gradients give (fp16 3.2e-4 and
    1.3e-2, bf16 2.6e-3 and 1e-1; outputs of a forward alone 6e-3 and 4e-2 at most)."""
    half = case["dtype"] == "float16"
    grads = case["kind"] in ("train", "varlen_train")
    return {"rel": 1.3e-3 if half else 1.0e-2,
            "max": (5.0e-2 if half else 4.0e-1) if grads else (2.5e-2 if half else 1.6e-1)}


def _attend64(q, k, v, causal, do=None):
    """One head in 64 bits: q [n, d], k and v [m, d] -> o, or (o, dq, dk, dv)."""
    scale = 1.0 / math.sqrt(q.shape[-1])
    s = (q @ k.T).mul_(scale)
    if causal:
        s.masked_fill_(torch.ones(s.shape, dtype=torch.bool, device=s.device).triu_(1), -math.inf)
    p = torch.softmax(s, dim=-1)
    del s
    o = p @ v
    if do is None:
        return o
    dv = p.T @ do
    ds = (do @ v.T).sub_((do * o).sum(-1, keepdim=True)).mul_(p).mul_(scale)
    return o, ds @ k, ds.T @ q, dv


def exact(case, seed):
    """What `run` returns, in 64 bits."""
    x = _inputs(case, seed)
    hq, hkv = case["heads_q"], case["heads_kv"]
    group = hq // hkv
    f64 = lambda t: t.double()
    if case["kind"] == "decode":
        out = torch.empty(x["q"].shape, dtype=torch.float64, device="cuda")
        for b, n in enumerate(_lengths(case)):
            for h in range(hkv):
                kv = [f64(t[b, :n, h] if case["layout"] == "bshd" else t[b, h, :n]) for t in (x["k"], x["v"])]
                sl = slice(h * group, (h + 1) * group)
                out[b, 0, sl] = _attend64(f64(x["q"][b, 0, sl]), *kv, False)
        return out
    # (rows of q, rows of k) as [n, heads, d] views, one per batch entry or segment
    if case["kind"] in ("prefill", "train"):
        parts = [(lambda t, b=b: t[b].transpose(0, 1)) for b in range(case["batch"])]
    else:
        ends = torch.tensor([0] + _lengths(case)).cumsum(0).tolist()
        parts = [(lambda t, a=a, e=e: t[a:e]) for a, e in zip(ends, ends[1:])]
    names = ["q", "k", "v"] + (["do"] if "do" in x else [])
    out = [torch.zeros(x[n].shape, dtype=torch.float64, device="cuda") for n in (["q"] + names[:3] if "do" in x else ["q"])]
    for part in parts:
        for h in range(hq):
            g = h // group
            q, k, v = f64(part(x["q"])[:, h]), f64(part(x["k"])[:, g]), f64(part(x["v"])[:, g])
            if "do" not in x:
                part(out[0])[:, h] = _attend64(q, k, v, case["causal"])
                continue
            o, dq, dk, dv = _attend64(q, k, v, case["causal"], f64(part(x["do"])[:, h]))
            part(out[0])[:, h] = o
            part(out[1])[:, h] = dq
            part(out[2])[:, g] += dk
            part(out[3])[:, g] += dv
    return out[0] if len(out) == 1 else tuple(out)
