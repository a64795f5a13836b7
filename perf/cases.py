"""The work of a user of this package, as cases that can be timed and compared.

A layer of a model uses the cache in two ways: it hands it a whole prompt once, and then one token after the other.
A case is one of

  prompt  a new cache takes a prompt of ``context`` tokens in one layer and then the first generated token: what the
          cache adds to the time to the first token
  token   one more token of a generation that is under way: the decode step of one layer with its attention
  fit     the factorisation of a prompt alone (``cast_lrqk_prefill``)

Head counts, head widths, ranks, active-set sizes and contexts are those of ``synth.WORKLOADS``, of the benchmark's
options and of the tests.  Prompts are low-rank plus noise with a rank above the factorisation's: a key matrix of
exactly that rank makes the r x r systems nearly singular, and then two correct implementations in the same
precision do not agree.

Outputs leave out the slots of the active set in their order (``Kgpu``, ``Vgpu``, the token ids): which slot a token
takes, and which of two tokens with nearly the same proxy score is in the set, follows the last bit of the factors.
The attention over the active set, which does not depend on the order, stands for it.
"""
import math

import torch

from lrqk_amd import DynamicLRQKCache, cast_lrqk_prefill, synth

DTYPES = {"bf16": torch.bfloat16, "fp32": torch.float32}
MORE_TOKENS = 32768   # room for generated tokens that a cache is created with
QUERY_SCALE = 4.0     # logits of a trained model spread over several units, so the attention has peaks
STREAM = 256          # generated tokens drawn ahead; a longer generation walks back and forth over them


def _case(name, kind, heads, kv_heads, head_dim, dtype, batch, context, r, k, lite, iters, tol):
    return {"name": name, "kind": kind, "heads": heads, "kv_heads": kv_heads, "head_dim": head_dim, "dtype": dtype,
            "batch": batch, "context": context, "r": r, "k": k, "lite": lite, "iters": iters, "tol": tol}


def listed():
    return [
        # short fp32 chat context of the 28 / 4 head shape: the smallest step, launches and host time count
        _case("token 4K fp32", "token", 28, 4, 128, "fp32", 1, 4096, 16, 512, 32, 1, 1e-2),
        # an ordinary long context of the 32 / 8 head shape
        _case("token 32K", "token", 32, 8, 128, "bf16", 1, 32768, 32, 2048, 64, 2, 1e-2),
        # the longest context the method is quoted on
        _case("token 128K", "token", 32, 8, 128, "bf16", 1, 131072, 32, 2048, 64, 2, 1e-2),
        # four sequences served together, as the full decoder steps them
        _case("token 4x64K", "token", 32, 8, 128, "bf16", 4, 65536, 32, 2048, 64, 2, 1e-2),
        # the throughput setting: small rank and active set, up to eight iterations
        _case("token 64K r16", "token", 32, 8, 128, "bf16", 1, 65536, 16, 1024, 16, 8, 1e-8),
        # the accuracy setting: large rank, active set and ring
        _case("token 64K r64", "token", 32, 8, 128, "bf16", 1, 65536, 64, 4096, 128, 4, 1e-10),
        # prompts of the same settings
        _case("prompt 4K fp32", "prompt", 28, 4, 128, "fp32", 1, 4096, 16, 512, 32, 1, 1e-2),
        # a batch of short prompts of odd length, narrow heads
        _case("prompt 3x2.5K d64", "prompt", 32, 8, 64, "bf16", 3, 2531, 16, 1024, 16, 2, 1e-2),
        _case("prompt 32K", "prompt", 32, 8, 128, "bf16", 1, 32768, 32, 2048, 64, 2, 1e-2),
        _case("prompt 128K", "prompt", 32, 8, 128, "bf16", 1, 131072, 32, 2048, 64, 2, 1e-2),
        _case("prompt 16K r64", "prompt", 32, 8, 128, "bf16", 1, 16384, 64, 4096, 128, 4, 1e-10),
        # the factorisation alone, as the benchmark times it
        _case("fit 32K", "fit", 32, 8, 128, "bf16", 1, 32768, 32, 2048, 64, 4, 1e-8),
    ]


def draw(rng):
    kind = rng.choice(("token", "token", "prompt", "prompt", "fit"))
    heads, kv_heads = rng.choice(((32, 8), (28, 4), (16, 8), (24, 3)))
    head_dim = rng.choice((128, 128, 128, 64))
    dtype = rng.choice(("bf16", "bf16", "bf16", "fp32"))
    r = rng.choice((8, 16, 16, 24, 32, 32, 32, 48, 64))
    k, lite = rng.choice(((512, 32), (1024, 16), (2048, 64), (2048, 64), (4096, 128)))
    iters, tol = rng.choice(((1, 1e-2), (2, 1e-2), (2, 1e-2), (4, 1e-10), (8, 1e-8)))
    low = 2 * k + lite
    # the passes over a prompt get longer with the rank, the iterations and the width of an element
    high = 131072 if dtype == "bf16" else 65536
    if kind != "token" and (r > 32 or dtype == "fp32" or head_dim != 128):
        high = 16384
    if kind != "token" and r > 32:
        iters = min(iters, 4)
    total = int(math.exp(rng.uniform(math.log(low), math.log(high))))
    batch = rng.choice([n for n in (1, 1, 1, 2, 3, 4) if total // n >= low])
    return {"kind": kind, "heads": heads, "kv_heads": kv_heads, "head_dim": head_dim, "dtype": dtype, "batch": batch,
            "context": total // batch, "r": min(r, head_dim // 2), "k": k, "lite": lite, "iters": iters, "tol": tol}


def _workload(case):
    return synth.Workload("case", case["heads"], case["kv_heads"], case["head_dim"], case["batch"],
                          DTYPES[case["dtype"]], case["context"], case["r"], case["k"], case["lite"],
                          (case["iters"],) * 2, (case["tol"],) * 2, 0, rho=3 * case["r"] // 2, sigma=0.05)


def _new_cache(w, more_tokens=MORE_TOKENS):
    return DynamicLRQKCache(r=w.r, num_active_tokens=w.num_active_tokens, max_iter=w.max_iter, lite_tokens=w.lite_tokens,
                            tol=w.tol, max_sequence_length=w.context + more_tokens, num_key_value_groups=w.groups)


class _Generation:
    """The tokens of a generation: queries that turn a little from one to the next, keys and values of the prompt's
    subspaces."""

    def __init__(self, w, q_last, bases, gen):
        queries = []
        q = q_last.float()
        for _ in range(STREAM):
            q = synth.rotate_query(gen, q)
            queries.append(q.to(w.dtype))
        keys, _ = synth.low_rank_noise(gen, w.batch, w.num_kv_heads, STREAM, w.head_dim, w.rho, w.sigma, w.dtype, bases[1])
        values, _ = synth.low_rank_noise(gen, w.batch, w.num_kv_heads, STREAM, w.head_dim, w.rho, w.sigma, w.dtype, bases[2])
        self.tokens = [(queries[t], keys[:, :, t:t + 1].contiguous(), values[:, :, t:t + 1].contiguous())
                       for t in range(STREAM)]
        self.at, self.step = 0, 1

    def next(self):
        token = self.tokens[self.at]
        if not 0 <= self.at + self.step < STREAM:
            self.step = -self.step
        self.at += self.step
        return token


def prepare(case, seed):
    w = _workload(case)
    q, k, v, bases, gen = synth.prompt_qkv(w, seed, device="cuda")
    q *= QUERY_SCALE
    if case["kind"] == "fit":
        return {"kind": "fit", "w": w, "seed": seed, "q": q, "k": k}
    if case["kind"] == "prompt":
        gen_q = synth.rotate_query(gen, q[:, :, -1:].float()).to(w.dtype)
        new = [synth.low_rank_noise(gen, w.batch, w.num_kv_heads, 1, w.head_dim, w.rho, w.sigma, w.dtype, b)[0]
               for b in bases[1:]]
        return {"kind": "prompt", "w": w, "seed": seed, "prompt": (q, k, v), "token": (gen_q, *new)}
    generation = _Generation(w, q[:, :, -1:], bases, gen)
    cache = _new_cache(w)
    torch.manual_seed(seed)
    cache.update(q, k, v, 0)
    cache.lwattn[0].attn_in_step = True
    for _ in range(4):   # a generation under way
        cache.update(*generation.next(), 0)
    return {"kind": "token", "cache": cache, "generation": generation}


def _step_outputs(engine):
    return {"attention": engine.last_attn, "q_hat": engine.last_q_hat, "k_hat": engine.last_k_hat, "B_Q": engine.B_Q,
            "B_K": engine.B_K}


def run(state):
    if state["kind"] == "token":
        cache = state["cache"]
        cache.update(*state["generation"].next(), 0)
        return _step_outputs(cache.lwattn[0])
    w = state["w"]
    torch.manual_seed(state["seed"])   # the initial factors are drawn from torch's generator
    if state["kind"] == "fit":
        return tuple(cast_lrqk_prefill(state["q"], state["k"], w.r, max_iter=w.max_iter[0], tol=w.tol[0]))
    cache = _new_cache(w, 1024)
    cache.update(*state["prompt"], 0)
    engine = cache.lwattn[0]
    engine.attn_in_step = True
    cache.update(*state["token"], 0)
    return {**_step_outputs(engine), "A_K": engine.A_K, "store": engine.KVcpu.tensor()}


def work(case):
    w = _workload(case)
    e = torch.empty((), dtype=w.dtype).element_size()
    bh, bkv, l, r, d = w.batch * w.num_heads, w.batch * w.num_kv_heads, w.context, w.r, w.head_dim
    n, iters = w.num_active_tokens + w.lite_tokens, w.max_iter[0]
    # a step: the key factors are scanned once, the active rows (K, V and factors) read once, B_Q and B_K read and written
    step_bytes = bh * e * (l * r + n * (2 * d + r) + 4 * r * d)
    step_flops = 2.0 * bh * (l * r + n * (2 * d + r * (r + d)) + iters * 2 * r * r)
    # a fit: Q and K are read once, the initial factors read and the factors written; every iteration forms two
    # products with Q and two with K and the r x r sums over each side
    fit_bytes = (bh + bkv) * l * d * e + 2 * bh * (l * r * (4 + e) + 2 * r * d * e)
    fit_flops = 2.0 * bh * l * r * (iters * 2 * (2 * d + r) + 2 * (d + r))
    if case["kind"] == "token":
        return {"bytes": step_bytes, "flops": step_flops}
    if case["kind"] == "fit":
        return {"bytes": fit_bytes, "flops": fit_flops}
    # a prompt: the fit (of A_Q only the last row is used), the scan of its proxy scores, K and V to the host store
    # (they cross the host link), the active rows
    prompt_bytes = fit_bytes - bh * l * r * e + bh * l * r * e + 3 * bkv * l * d * e + 4 * bh * n * d * e
    return {"bytes": prompt_bytes + step_bytes, "flops": fit_flops + 2.0 * bh * l * r + step_flops}


def tolerance(case):
    # Worst output over the listed and some drawn cases.  bf16: 2.9e-3 between a run whose factors come from the
    # row-by-row formulation and one on Gram matrices (a factor that rounds to the other neighbour moves the proxy
    # scores, and with them a few tokens at the edge of the active set); 1.4e-3 between an fp32 and an fp64 step.
    # fp32: a plain fp32 evaluation of the factorisation is up to 7e-5 off its fp64 evaluation (ranks 8 to 64).
    return {"rel": 1e-2 if case["dtype"] == "bf16" else 2e-4}
