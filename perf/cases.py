"""The work that a program built on this framework has it do, case by case: single linear layers,
decode and prefill attention, the decode step of one sequence and of a batch, and prompt prefill,
over the sizes of the configurations in llamatov_amd/model.py and of the benchmark.

Inputs, weights included, are made on the GPU from the seed.  Device memory that the engine owns is
returned as torch views of its buffers (no copy)."""
from __future__ import annotations

import ctypes
import math

import numpy as np
import torch

from llamatov_amd import engine, model
from llamatov_amd._lib import LT_KV_F16, LT_KV_F32, call

F64 = torch.float64

# widths of the two architectures in llamatov_amd/model.py (vocab 0: the full vocabulary;
# 4096 is the small test configuration's)
CFG = {"0.5b": model.QWEN25_05B, "8b": model.LLAMA3_8B}


def listed():
    return [
        # the feed-forward input matrix of the 0.5B model, one token: the smallest call that a
        # kernel-per-op program makes (quantize the row, then the GEMV)
        {"name": "linear-ffn-0.5b", "kind": "linear", "N": 4864, "K": 896, "planar": False, "resid": False},
        # the vocabulary projection of the 8B model, one token, over the planar copy
        {"name": "linear-head-8b", "kind": "linear", "N": 128256, "K": 4096, "planar": True, "resid": False},
        # greedy decode of one short conversation on the 0.5B model, an id read back per token
        {"name": "decode-0.5b", "kind": "decode", "model": "0.5b", "layers": 24, "vocab": 0, "ctx": 61, "tokens": 8,
         "kv": "f16", "nsplit": 1, "top_k": 0},
        # the same with the sampler, some turns later
        {"name": "decode-0.5b-sampled", "kind": "decode", "model": "0.5b", "layers": 24, "vocab": 0, "ctx": 301,
         "tokens": 8, "kv": "f16", "nsplit": 1, "top_k": 40},
        # near the end of the 1024-token context, with the default profile's fp32 cache
        {"name": "decode-0.5b-long", "kind": "decode", "model": "0.5b", "layers": 24, "vocab": 0, "ctx": 905,
         "tokens": 8, "kv": "f32", "nsplit": 1, "top_k": 0},
        # the 8B model's layers (two of its 32) after a 512-token prompt, context split 16 ways
        {"name": "decode-8b", "kind": "decode", "model": "8b", "layers": 2, "vocab": 4096, "ctx": 512, "tokens": 16,
         "kv": "f16", "nsplit": 16, "top_k": 0},
        # batched serving at the 0.5B widths (four layers): a few and many sequences of unequal lengths
        {"name": "batch-8", "kind": "batch", "model": "0.5b", "layers": 4, "vocab": 4096, "B": 8, "ctx": 700,
         "tokens": 4, "kv": "f16"},
        {"name": "batch-64", "kind": "batch", "model": "0.5b", "layers": 4, "vocab": 4096, "B": 64, "ctx": 500,
         "tokens": 4, "kv": "f16"},
        # a prompt on the whole 0.5B model, an odd length, one split (the default)
        {"name": "prefill-0.5b", "kind": "prefill", "model": "0.5b", "layers": 24, "vocab": 0, "T": 509, "kv": "f16",
         "nsplit": 1},
        # the benchmark's 512-token prompt on the 8B model's layers (two of them)
        {"name": "prefill-8b", "kind": "prefill", "model": "8b", "layers": 2, "vocab": 4096, "T": 512, "kv": "f16",
         "nsplit": 16},
        # decode attention over a long cache (the benchmark's 32 q / 8 KV heads of 128)
        {"name": "attn-decode-16k", "kind": "attn", "B": 1, "L": 16384, "nh": 32, "nkv": 8, "hd": 128, "kv": "f16"},
        # causal attention of a long prompt at the 8B geometry
        {"name": "attn-prefill-2k", "kind": "causal", "T": 2048, "past": 0, "nh": 32, "nkv": 8, "hd": 128,
         "kv": "f16", "nsplit": 1},
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["linear", "decode", "decode", "batch", "prefill", "prefill", "attn", "causal"])
    kv = rng.choice(["f16", "f16", "f32"])
    if kind == "linear":
        N, K = rng.choice([(4864, 896), (896, 4864), (1152, 896), (4096, 4096), (14336, 4096), (4096, 14336),
                           (6144, 4096), (128256, 4096), (151936, 896)])
        N = N if rng.random() < 0.5 else max(8, N - rng.randrange(1, 64))
        return {"kind": kind, "N": N, "K": K, "planar": K % 1024 == 0 and rng.random() < 0.5,
                "resid": rng.random() < 0.5}
    if kind == "decode":
        if rng.random() < 0.6:
            return {"kind": kind, "model": "0.5b", "layers": 24, "vocab": 0, "ctx": _log_int(rng, 4, 1000),
                    "tokens": 8, "kv": kv, "nsplit": 1, "top_k": rng.choice([0, 0, 20, 40, 200])}
        return {"kind": kind, "model": "8b", "layers": 2, "vocab": 4096, "ctx": _log_int(rng, 16, 1000),
                "tokens": 8, "kv": kv, "nsplit": rng.choice([1, 8, 16, 16]), "top_k": 0}
    if kind == "batch":
        return {"kind": kind, "model": "0.5b", "layers": 4, "vocab": 4096, "B": _log_int(rng, 2, 64),
                "ctx": _log_int(rng, 24, 700), "tokens": 4, "kv": kv}
    if kind == "prefill":
        if rng.random() < 0.5:
            return {"kind": kind, "model": "0.5b", "layers": 24, "vocab": 0, "T": _log_int(rng, 7, 509), "kv": kv,
                    "nsplit": 1}
        return {"kind": kind, "model": "8b", "layers": 2, "vocab": 4096, "T": _log_int(rng, 7, 512), "kv": kv,
                "nsplit": rng.choice([1, 16])}
    nh, nkv, hd = rng.choice([(32, 8, 128), (32, 8, 128), (14, 2, 64)])
    if kind == "attn":
        B = rng.choice([1, 1, 2, 4, 8])
        return {"kind": kind, "B": B, "L": _log_int(rng, 300, 32768 // B), "nh": nh, "nkv": nkv, "hd": hd, "kv": kv}
    T = _log_int(rng, 16, 1500)
    return {"kind": kind, "T": T, "past": rng.choice([0, 0, rng.randrange(1, 512)]), "nh": nh, "nkv": nkv, "hd": hd,
            "kv": kv, "nsplit": rng.choice([1, 1, 8])}


# ---- inputs ------------------------------------------------------------------------------------
def _gen(seed, what):
    g = torch.Generator(device="cuda")
    g.manual_seed((int(seed) * 1000003 + what) & 0x7FFFFFFFFFFFFFFF)
    return g


def _normal(seed, what, *shape, std=1.0):
    return torch.randn(*shape, generator=_gen(seed, what), device="cuda") * std


def _q8(seed, what, N, K):
    """An N x K matrix of N(0, 0.02) as GGUF Q8_0 blocks: uint8 [N, K/32*34]."""
    w = _normal(seed, what, N, K, std=0.02).view(N, K // 32, 32)
    amax = w.abs().amax(-1)
    d = torch.where(amax > 0, amax / 127, torch.ones_like(amax)).half()
    q = torch.round(w / d.float()[..., None]).clamp_(-127, 127).to(torch.int8)
    return torch.cat([d[..., None].view(torch.uint8), q.view(torch.uint8)], -1).view(N, -1)


def _q8_values(blocks):
    """The float64 values of Q8_0 blocks."""
    b = blocks.view(blocks.shape[0], -1, 34)
    d = b[..., :2].contiguous().view(torch.float16).to(F64)
    return (b[..., 2:].contiguous().view(torch.int8).to(F64) * d).view(blocks.shape[0], -1)


def _config(case):
    c = CFG[case["model"]]
    ctx = 1024 if case["kind"] != "batch" else 768
    return c.replace(n_layers=case["layers"], vocab=case["vocab"] or c.vocab, tied=True, max_ctx=ctx)


def _weights(case, seed):
    """GGUF-named tensors on the GPU: Q8_0 blocks, norm weights near 1, q/k/v biases."""
    c = _config(case)
    E, F, Q, KV = c.n_embd, c.n_ff, c.n_head * c.head_dim, c.n_head_kv * c.head_dim
    w = {"token_embd.weight": _q8(seed, 1, c.vocab, E), "output_norm.weight": 1 + _normal(seed, 2, E, std=0.1)}
    for il in range(c.n_layers):
        p, s = "blk.%d." % il, 100 * (il + 1)
        w[p + "attn_norm.weight"] = 1 + _normal(seed, s, E, std=0.1)
        w[p + "ffn_norm.weight"] = 1 + _normal(seed, s + 1, E, std=0.1)
        for k, (name, N, K) in enumerate([("attn_q", Q, E), ("attn_k", KV, E), ("attn_v", KV, E),
                                          ("attn_output", E, Q), ("ffn_gate", F, E), ("ffn_up", F, E),
                                          ("ffn_down", E, F)]):
            w[p + name + ".weight"] = _q8(seed, s + 2 + k, N, K)
        if c.qkv_bias:
            for k, (name, N) in enumerate([("attn_q", Q), ("attn_k", KV), ("attn_v", KV)]):
                w[p + name + ".bias"] = _normal(seed, s + 10 + k, N, std=0.02)
    return c, w


def _token_ids(seed, what, n, vocab):
    return [int(t) for t in torch.randint(0, vocab, (n,), generator=_gen(seed, what), device="cuda").tolist()]


def _batch_lengths(case):
    """Prompt lengths of a batch, spread over ctx/8 .. ctx."""
    return [max(1, int(case["ctx"] * (0.125 + 0.875 * (0.618034 * (b + 1) % 1)))) for b in range(case["B"])]


class _Held:
    """What a program keeps: freed when nothing refers to it any more."""

    def __init__(self):
        self.parts = []

    def keep(self, x):
        self.parts.append(x)
        return x

    def __del__(self):
        try:
            engine.get_device().sync()
            for x in reversed(self.parts):
                x.free()
        except Exception:
            pass


class _Memory:
    def __init__(self, held, ptr, shape, typestr):
        self.held = held
        self.__cuda_array_interface__ = {"shape": tuple(shape), "typestr": typestr, "data": (int(ptr), False),
                                         "version": 3, "strides": None}


def _view(held, ptr, shape, typestr):
    """A torch tensor over device memory that `held` owns."""
    return torch.as_tensor(_Memory(held, ptr, shape, typestr), device="cuda")


def _dev(t, dtype=np.float32):
    return engine.DevTensor(t.data_ptr(), t.shape, dtype, owns=False)


def _kv(case):
    return (LT_KV_F16, torch.float16, "<f2") if case["kv"] == "f16" else (LT_KV_F32, torch.float32, "<f4")


def _resident(case, seed, held):
    c, w = _weights(case, seed)
    torch.cuda.synchronize()
    return c, held.keep(engine.ResidentModel(c, {k: v.cpu().numpy() for k, v in w.items()}, layouts="fused"))


def prepare(case, seed):
    return globals()["_prepare_" + case["kind"]](case, seed)


def run(state):
    return state["run"](state)


# ---- one linear layer: quantize the activation row, then the Q8_0 GEMV --------------------------
def _linear_inputs(case, seed):
    N, K = case["N"], case["K"]
    return _q8(seed, 1, N, K), _normal(seed, 2, K), _normal(seed, 3, N) if case["resid"] else None


def _prepare_linear(case, seed):
    N, K = case["N"], case["K"]
    W, x, r = _linear_inputs(case, seed)
    y = torch.empty(N, device="cuda")
    xq, xd = torch.empty(K, dtype=torch.int8, device="cuda"), torch.empty(K // 32, dtype=torch.int16, device="cuda")
    if case["planar"]:
        P = torch.empty_like(W)
        torch.cuda.synchronize()
        call("lt_q8_to_planar", engine.get_device().handle, engine._vp(W.data_ptr()), engine._vp(P.data_ptr()), N, K)
        engine.get_device().sync()
        W = P
    return {"run": _run_linear_planar if case["planar"] else _run_linear, "keep": (W, x, r, y, xq, xd), "y": y,
            "W": engine.Q8Weight(None, K, t=_dev(W, np.uint8), N=N), "x": _dev(x), "out": _dev(y),
            "xq": _dev(xq, np.int8), "xd": _dev(xd, np.uint16), "r": None if r is None else _dev(r)}


def _run_linear(s):
    if s["r"] is None:
        engine.q8_linear_into(s["x"], s["W"], s["out"], s["xq"], s["xd"])
    else:
        engine.q8_linear_add_residual_into(s["x"], s["W"], s["r"], s["out"], s["xq"], s["xd"])
    return s["y"]


def _run_linear_planar(s):
    W = s["W"]
    engine.quant_q8_into(s["x"], s["xq"], s["xd"], W.K)
    call("lt_q8_gemv_pl", W.t.dev.handle, W.t.vp, s["xq"].vp, s["xd"].vp, engine._vp(s["r"]), s["out"].vp, W.N, W.K)
    return s["y"]


# ---- one sequence's decode: ids chosen by the host, one graph replay and one id back per token --
def _prepare_decode(case, seed):
    held = _Held()
    c, m = _resident(case, seed, held)
    kv, _, ts = _kv(case)
    plan = held.keep(engine.DecodePlan(m, engine.Profile(kv_dtype=kv, attn_nsplit=case["nsplit"])))
    if case["top_k"]:
        plan.set_sampling(0.8, case["top_k"], 0.95, seed=seed)
    ctx, n = case["ctx"], case["tokens"]
    graph = held.keep(engine.StepGraph(plan))
    graph.seed(_token_ids(seed, 11, ctx, c.vocab), batched=True)
    graph.capture()
    out = [_view(held, plan.logits.ptr, (c.vocab,), "<f4")]
    for cache in plan.caches:
        out += [_view(held, t.ptr, (ctx + n, c.kv_dim), ts) for t in (cache.k, cache.v)]
    return {"run": _run_decode, "held": held, "plan": plan, "graph": graph, "out": out, "ctx": ctx,
            "lens": np.full(c.n_layers, ctx, np.int32), "ids": _token_ids(seed, 12, n, c.vocab)}


def _run_decode(s):
    plan = s["plan"]
    plan.dev.h2d(plan.lens.ptr, s["lens"])   # back to the end of the prompt
    for cache in plan.caches:
        cache.length = s["ctx"]
    return [s["graph"].replay_token(t) for t in s["ids"]], s["out"]


# ---- a batch of sequences, one token of each per step -------------------------------------------
def _prepare_batch(case, seed):
    held = _Held()
    c, m = _resident(case, seed, held)
    kv, _, ts = _kv(case)
    B, n = case["B"], case["tokens"]
    plan = held.keep(engine.BatchDecodePlan(m, B, engine.Profile(kv_dtype=kv)))
    lens = _batch_lengths(case)
    for b in range(B):
        plan.prefill(b, _token_ids(seed, 1000 + b, lens[b], c.vocab))
    graph = held.keep(engine.BatchStepGraph(plan))
    graph.capture()
    out = [_view(held, plan.logits.ptr, (B, c.vocab), "<f4")]
    # the first and last layers' cache rows of the first and last sequences
    rows = [(il, t.ptr + b * plan.slot_bytes, lens[b] + n) for il in (0, c.n_layers - 1) for b in (0, B - 1)
            for t in (plan.k[il], plan.v[il])]
    out += [_view(held, p, (L, c.kv_dim), ts) for _, p, L in rows]
    return {"run": _run_batch, "held": held, "plan": plan, "graph": graph, "out": out, "length": lens,
            "lens": np.array(lens + [L + 1 for L in lens], np.int32),
            "ids": [_token_ids(seed, 12 + i, B, c.vocab) for i in range(n)]}


def _run_batch(s):
    plan, got = s["plan"], []
    plan.dev.h2d(plan.lens.ptr, s["lens"])   # back to the ends of the prompts
    plan.length = list(s["length"])
    for ids in s["ids"]:
        plan.set_tokens(ids)
        s["graph"].replay()
        got.append(plan.read_tokens())
    return np.array(got), s["out"]


# ---- a prompt -----------------------------------------------------------------------------------
def _prepare_prefill(case, seed):
    held = _Held()
    c, m = _resident(case, seed, held)
    kv, _, ts = _kv(case)
    plan = held.keep(engine.DecodePlan(m, engine.Profile(kv_dtype=kv, attn_nsplit=case["nsplit"])))
    m.prefill_tiles()
    plan.prefill_buffers(case["T"])
    out = [_view(held, plan.logits.ptr, (c.vocab,), "<f4")]
    for cache in plan.caches:
        out += [_view(held, t.ptr, (case["T"], c.kv_dim), ts) for t in (cache.k, cache.v)]
    return {"run": _run_prefill, "held": held, "plan": plan, "out": out,
            "ids": _token_ids(seed, 11, case["T"], c.vocab)}


def _run_prefill(s):
    s["plan"].reset()
    engine.forward_prefill(s["plan"], s["ids"])
    return s["plan"].read_token(), s["out"]


# ---- decode attention over a cache --------------------------------------------------------------
def _attn_inputs(case, seed):
    kv = _kv(case)[1]
    B, L, W = case["B"], case["L"], case["nkv"] * case["hd"]
    q = _normal(seed, 1, B, case["nh"] * case["hd"])
    k, v = (_normal(seed, s, B, L, W).to(kv) for s in (2, 3))
    lens = [L - (b * L) // (2 * B) for b in range(B)]
    return q, k, v, lens


def _prepare_attn(case, seed):
    q, k, v, lens = _attn_inputs(case, seed)
    B, nh, hd = case["B"], case["nh"], case["hd"]
    nsplit = engine.attn_nsplit_for(B, case["L"], case["nkv"])
    out = torch.empty_like(q)
    n = int(engine._lib.raw("lt_attn_workspace_size")(B, nh, hd, nsplit))
    ws = torch.empty(max(1, n), dtype=torch.uint8, device="cuda")
    ld = torch.tensor(lens, dtype=torch.int32, device="cuda")
    p = [engine._vp(t.data_ptr()) for t in (q, k, v, ld, out)]
    return {"run": _run_attn, "keep": (q, k, v, ld, ws), "y": out,
            "args": (engine.get_device().handle, *p, B, nh, case["nkv"], hd, ctypes.c_float(hd ** -0.5), case["L"],
                     nsplit, _kv(case)[0], engine._vp(ws.data_ptr()), n)}


def _run_attn(s):
    call("lt_attn_decode", *s["args"])
    return s["y"]


# ---- causal attention of a prompt ---------------------------------------------------------------
def _causal_inputs(case, seed):
    kv = _kv(case)[1]
    T, W = case["T"], case["nkv"] * case["hd"]
    n = T + case["past"]
    # q rows lie in the q|k|v rows of the projection
    qkv = _normal(seed, 1, T, case["nh"] * case["hd"] + 2 * W)
    k, v = (_normal(seed, s, n, W).to(kv) for s in (2, 3))
    return qkv, k, v


def _prepare_causal(case, seed):
    qkv, k, v = _causal_inputs(case, seed)
    T, nh, hd = case["T"], case["nh"], case["hd"]
    out = torch.empty(T, nh * hd, device="cuda")
    n = int(engine._lib.raw("lt_attn_workspace_size")(T, nh, hd, case["nsplit"]))
    ws = torch.empty(max(1, n), dtype=torch.uint8, device="cuda")
    past = torch.tensor([case["past"]], dtype=torch.int32, device="cuda")
    a = [engine._vp(t.data_ptr()) for t in (k, v, past, out)]
    return {"run": _run_causal, "keep": (qkv, k, v, past, ws), "y": out,
            "args": (engine.get_device().handle, engine._vp(qkv.data_ptr()), qkv.shape[1], *a, T, nh, case["nkv"], hd,
                     ctypes.c_float(hd ** -0.5), T + case["past"], case["nsplit"], _kv(case)[0],
                     engine._vp(ws.data_ptr()), n)}


def _run_causal(s):
    call("lt_attn_prefill", *s["args"])
    return s["y"]


# ---- what a pass cannot do without --------------------------------------------------------------
def _step_work(case, c, tokens, attended, streams):
    """tokens through every layer and `streams` of them through the head, the weights read
    `streams` times, `attended` query-key pairs in each layer."""
    E, F, Q, KV = c.n_embd, c.n_ff, c.q_dim, c.kv_dim
    layer, head = c.n_qkv * E + E * Q + 3 * F * E, c.vocab * E
    return {"weights": (c.n_layers * layer + head) * 34 / 32,
            "flops": 2 * c.n_layers * (tokens * layer + 2 * attended * Q) + 2 * streams * head}


def work(case):
    esz = 2 if case.get("kv") == "f16" else 4
    kind = case["kind"]
    if kind == "linear":
        N, K = case["N"], case["K"]
        return {"bytes": N * K * 34 / 32 + 4 * K + 4 * N * (2 if case["resid"] else 1), "flops": 2 * N * K}
    if kind == "attn":
        n = sum(case["L"] - (b * case["L"]) // (2 * case["B"]) for b in range(case["B"]))
        Q = case["nh"] * case["hd"]
        return {"bytes": 2 * n * case["nkv"] * case["hd"] * esz + 8 * case["B"] * Q, "flops": 4 * n * Q}
    if kind == "causal":
        T, n, Q = case["T"], case["T"] + case["past"], case["nh"] * case["hd"]
        return {"bytes": 2 * n * case["nkv"] * case["hd"] * esz + 8 * T * Q,
                "flops": 4 * Q * (T * case["past"] + T * (T + 1) // 2)}
    c = _config(case)
    row = 2 * c.n_layers * c.kv_dim * esz   # one position's K and V in every layer
    if kind == "prefill":
        T = case["T"]
        w = _step_work(case, c, T, T * (T + 1) // 2, 1)
        return {"bytes": w["weights"] + row * T + 4 * c.vocab, "flops": w["flops"]}
    n = case["tokens"]
    if kind == "decode":
        pairs = sum(case["ctx"] + i + 1 for i in range(n))
        w = _step_work(case, c, n, pairs, n)
        return {"bytes": n * (w["weights"] + 4 * c.vocab) + row * pairs, "flops": w["flops"]}
    pairs = sum(L + i + 1 for L in _batch_lengths(case) for i in range(n))
    w = _step_work(case, c, n * case["B"], pairs, n * case["B"])
    return {"bytes": n * (w["weights"] + 4 * c.vocab * case["B"]) + row * pairs, "flops": w["flops"]}


# ---- the same in 64 bits ------------------------------------------------------------------------
def _quant64(x):
    """Q8_0 activation quantization over the last axis, the values it leaves."""
    b = x.view(*x.shape[:-1], -1, 32)
    amax = b.abs().amax(-1, keepdim=True)
    d = (amax / 127).to(torch.float16).to(F64)
    d = torch.where(amax > 0, d, torch.ones_like(d))
    return (torch.round(b / d).clamp(-127, 127) * d).view(x.shape)


def _attention64(q, k, v, past):
    """q [T, nh, hd], k / v [past + T, nkv, hd]; row t attends past + t + 1 positions."""
    T, nh, hd = q.shape
    g = nh // k.shape[1]
    out = torch.empty_like(q)
    keep = torch.arange(k.shape[0], device=q.device)[None, :] <= past + torch.arange(T, device=q.device)[:, None]
    for h in range(nh):
        s = (q[:, h] @ k[:, h // g].t().contiguous()) * hd ** -0.5
        out[:, h] = torch.softmax(s.masked_fill(~keep, -math.inf), -1) @ v[:, h // g].contiguous()
    return out


def _rope64(x, pos, theta):
    hd = x.shape[-1]
    f = theta ** (-2.0 * torch.arange(hd // 2, dtype=F64, device=x.device) / hd)
    # the engine's table holds each frequency rounded to 32 bits, and the angle is a 32-bit product
    a = (pos[:, None].float() * f.float()).to(F64)[:, None, :]
    x1, x2 = x[..., : hd // 2], x[..., hd // 2:]
    return torch.cat([x1 * a.cos() - x2 * a.sin(), x1 * a.sin() + x2 * a.cos()], -1)


def _model64(c, w, ids, kv):
    """logits of the last position, [K, V] rows of every layer, for one sequence."""
    pos = torch.arange(len(ids), device="cuda")
    x = _q8_values(w["token_embd.weight"][torch.tensor(ids, device="cuda")])
    T, hd = len(ids), c.head_dim
    caches = []

    def norm(x, g):
        return _quant64(x * torch.rsqrt((x * x).mean(-1, keepdim=True) + c.norm_eps) * g.to(F64))

    def lin(x, name):
        y = x @ _q8_values(w[name + ".weight"]).t()
        return y + w[name + ".bias"].to(F64) if name + ".bias" in w else y

    for il in range(c.n_layers):
        p = "blk.%d." % il
        h = norm(x, w[p + "attn_norm.weight"])
        q = _rope64(lin(h, p + "attn_q").view(T, c.n_head, hd), pos, c.rope_theta)
        k = _rope64(lin(h, p + "attn_k").view(T, c.n_head_kv, hd), pos, c.rope_theta).to(kv).to(F64)
        v = lin(h, p + "attn_v").view(T, c.n_head_kv, hd).to(kv).to(F64)
        caches += [k.reshape(T, -1), v.reshape(T, -1)]
        x = x + lin(_quant64(_attention64(q, k, v, 0).reshape(T, -1)), p + "attn_output")
        h = norm(x, w[p + "ffn_norm.weight"])
        g, u = lin(h, p + "ffn_gate"), lin(h, p + "ffn_up")
        x = x + lin(_quant64(g / (1 + torch.exp(-g)) * u), p + "ffn_down")
    return norm(x[-1:], w["output_norm.weight"])[0] @ _q8_values(w["token_embd.weight"]).t(), caches


def exact(case, seed):
    kind, kv = case["kind"], _kv(case)[1] if "kv" in case else None
    if kind == "linear":
        W, x, r = _linear_inputs(case, seed)
        y = _q8_values(W) @ _quant64(x.to(F64))
        return y if r is None else y + r.to(F64)
    if kind == "attn":
        q, k, v, lens = _attn_inputs(case, seed)
        B, nh, nkv, hd = case["B"], case["nh"], case["nkv"], case["hd"]
        return torch.stack([_attention64(q[b].to(F64).view(1, nh, hd), k[b, :L].to(F64).view(L, nkv, hd),
                                         v[b, :L].to(F64).view(L, nkv, hd), L - 1).view(-1)
                            for b, L in enumerate(lens)])
    if kind == "causal":
        qkv, k, v = _causal_inputs(case, seed)
        T, nh, nkv, hd = case["T"], case["nh"], case["nkv"], case["hd"]
        n = T + case["past"]
        return _attention64(qkv[:, : nh * hd].to(F64).reshape(T, nh, hd), k.to(F64).view(n, nkv, hd),
                            v.to(F64).view(n, nkv, hd), case["past"]).view(T, -1)
    c, w = _weights(case, seed)
    if kind == "decode":
        ids = _token_ids(seed, 11, case["ctx"], c.vocab) + _token_ids(seed, 12, case["tokens"], c.vocab)
        logits, caches = _model64(c, w, ids, kv)
        return None, [logits] + caches   # the ids follow from each step's logits, or from the sampler
    if kind == "prefill":
        logits, caches = _model64(c, w, _token_ids(seed, 11, case["T"], c.vocab), kv)
        return None, [logits] + caches
    B, lens = case["B"], _batch_lengths(case)
    steps = [_token_ids(seed, 12 + i, B, c.vocab) for i in range(case["tokens"])]
    got = [_model64(c, w, _token_ids(seed, 1000 + b, lens[b], c.vocab) + [t[b] for t in steps], kv)
           for b in range(B)]
    rows = [got[b][1][2 * il + j] for il in (0, c.n_layers - 1) for b in (0, B - 1) for j in (0, 1)]
    return None, [torch.stack([g[0] for g in got])] + rows


def tolerance(case):
    # about four times the error measured against exact()
    if case["kind"] == "linear":
        return {"rel": 7e-7, "max": 2e-5}   # 32-bit sums of exact block dots (2e-7)
    if case["kind"] in ("attn", "causal"):
        return {"rel": 2e-6, "max": 1e-4}   # 32-bit dots, exponentials and sums (5e-7)
    # a difference of one rounding moves activation quants and travels through the layers after
    # it: 0.011 to 0.018 after one layer, 0.02 to 0.03 after 24
    return {"rel": 0.03, "max": 0.5, "differ": 0.01}
