"""The work this framework is timed on: what a llama.cpp user has the MI355X kernels do, through the public entry points.

Five kinds of call, each over the range of sizes it meets in use (sizes: the Llama-3-8B and Mixtral-8x7B shapes of the benchmark and
the tests, neighbours of them, and generic ones):

  mm       mi355.mul_mat: quantized weights x f32 activation rows.  One row is single-stream decoding, 2..32 rows are parallel
           sequences and speculative drafts, more are prompt batches.  All ten weight types.
  mmid     mi355.mul_mat_id: the routed expert products of a mixture-of-experts layer (8 experts of which each token uses 2).
  fa       mi355.flash_attn_ext: attention of one decoded token over a long f16 cache, or of a prompt batch under the causal mask,
           grouped-query heads, the cache laid out [cell][kv head][head size] as llama.cpp keeps it.
  fa_kv    mi355_flash_attn_ext_kv: one decoded token over a Q8_0 or Q4_0 cache (-ctk / -ctv q8_0, q4_0) read where it lies.
  decode   one token through the whole decoder stack (LlamaRunner.forward, replayed as a HIP graph as the benchmark does).
  prefill  one prompt batch through the whole decoder stack (LlamaRunner.forward), logits of the last token.
"""
import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.getcwd(), "llama.cpp_amd"))
import mi355  # noqa: E402
from mi355 import llama_graph as lg  # noqa: E402

TYPES = ("q4_0", "q4_1", "q5_0", "q5_1", "q8_0", "iq4_nl", "q4_K", "q5_K", "q6_K", "iq4_xs")
MOST = 14336 * 4096 * 1024                          # multiply-adds of the largest drawn product
SUPER = ("q4_K", "q5_K", "q6_K", "iq4_xs")          # blocks of 256; the others have blocks of 32


def listed():
    return [
        # one decoded token: an attention projection of an 8B model (the smallest call: launches and host work count)
        {"name": "mm q4_K 4096x4096 b1", "kind": "mm", "type": "q4_K", "N": 4096, "K": 4096, "B": 1},
        # eight parallel sequences through the feed-forward matrix of a larger model
        {"name": "mm q8_0 28672x8192 b8", "kind": "mm", "type": "q8_0", "N": 28672, "K": 8192, "B": 8},
        # a short prompt (or 64 parallel sequences) through the feed-forward matrix of the 8B model
        {"name": "mm q4_K 14336x4096 b64", "kind": "mm", "type": "q4_K", "N": 14336, "K": 4096, "B": 64},
        # a prompt batch of llama.cpp's default micro-batch size, per-32-block weights
        {"name": "mm q4_0 14336x4096 b512", "kind": "mm", "type": "q4_0", "N": 14336, "K": 4096, "B": 512},
        # the ragged end of a prompt on the down projection of a 7B model: 43 super-blocks per row, rows that start at any even byte
        {"name": "mm q6_K 4096x11008 b333", "kind": "mm", "type": "q6_K", "N": 4096, "K": 11008, "B": 333},
        # experts of the Mixtral-8x7B shape, a prompt batch
        {"name": "mmid q4_K 8x14336x4096 t512", "kind": "mmid", "type": "q4_K", "N": 14336, "K": 4096, "E": 8, "used": 2, "T": 512},
        # long-context decoding over an f16 cache
        {"name": "fa 1x32768 d128", "kind": "fa", "D": 128, "H": 32, "HK": 8, "Nq": 1, "Nkv": 32768},
        # a prompt batch that continues a conversation of some thousand tokens
        {"name": "fa 512x4096 d128", "kind": "fa", "D": 128, "H": 32, "HK": 8, "Nq": 512, "Nkv": 4096},
        # the first batch of a prompt, head size 80
        {"name": "fa 512x512 d80", "kind": "fa", "D": 80, "H": 32, "HK": 32, "Nq": 512, "Nkv": 512},
        # decoding at a medium context over a Q8_0 cache
        {"name": "fa_kv q8_0 1x8192 d128", "kind": "fa_kv", "cache": "q8_0", "D": 128, "H": 32, "HK": 8, "Nkv": 8192},
        # the headline figures of the benchmark: a token and a 512-token prompt of a Llama-3-8B-shaped Q4_K_M model
        {"name": "decode 8b q4_k_m kv512", "kind": "decode", "ftype": "q4_k_m", "layers": 32, "embd": 4096, "ff": 14336, "H": 32, "HK": 8, "vocab": 128256, "n_kv": 512},
        {"name": "prefill 8b q4_k_m t512", "kind": "prefill", "ftype": "q4_k_m", "layers": 32, "embd": 4096, "ff": 14336, "H": 32, "HK": 8, "vocab": 128256, "T": 512,
         "n_kv": 512},
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(("mm", "mm", "mm", "mmid", "fa", "fa", "fa_kv", "decode", "prefill"))
    if kind == "mm":
        t = rng.choice(TYPES)
        K = 256 * _log_int(rng, 4, 56)
        if t not in SUPER and rng.random() < 0.3:
            K += 32 * rng.randrange(1, 8)
        N, B = _log_int(rng, 1024, 32768), _log_int(rng, 1, 1024)
        return {"kind": kind, "type": t, "N": N, "K": K, "B": max(1, min(B, MOST // (N * K)))}
    if kind == "mmid":
        t = rng.choice(TYPES)
        N, K, T = 32 * _log_int(rng, 32, 448), 256 * _log_int(rng, 4, 32), _log_int(rng, 1, 768)
        return {"kind": kind, "type": t, "N": N, "K": K, "E": rng.choice((4, 8, 16)), "used": 2, "T": max(1, min(T, MOST // (2 * N * K)))}
    if kind == "fa":
        D, HK, g = rng.choice((64, 80, 128, 128, 256)), rng.choice((4, 8)), rng.choice((1, 4, 4, 8))
        if rng.random() < 0.5:
            return {"kind": kind, "D": D, "H": HK * g, "HK": HK, "Nq": 1, "Nkv": 32 * _log_int(rng, 8, 2048)}
        Nq = _log_int(rng, 33, 2048)
        return {"kind": kind, "D": D, "H": HK * g, "HK": HK, "Nq": Nq, "Nkv": (Nq + 31) // 32 * 32 + 32 * _log_int(rng, 1, 128)}
    if kind == "fa_kv":
        HK, g = rng.choice((4, 8)), rng.choice((1, 4, 8))
        return {"kind": kind, "cache": rng.choice(("q8_0", "q4_0")), "D": 128, "H": HK * g, "HK": HK, "Nkv": 256 * _log_int(rng, 1, 256)}
    embd = rng.choice((2048, 4096))
    c = {"kind": kind, "ftype": rng.choice(("q4_k_m", "q4_k_m", "q8_0", "q4_0")), "layers": _log_int(rng, 4, 24), "embd": embd, "ff": rng.choice((2, 3)) * embd + rng.choice((0, 2048)),
         "H": embd // 128, "HK": rng.choice((4, 8)), "vocab": rng.choice((32000, 128256))}
    if kind == "decode":
        c["n_kv"] = 256 * _log_int(rng, 1, 32)
    else:
        c["T"] = _log_int(rng, 33, 768)
        c["n_kv"] = (c["T"] + 255) // 256 * 256 + 256 * rng.choice((0, 0, 1, 4))
    return c


# ---------------------------------------------------------------------------------------------- inputs
def _gen(seed):
    return torch.Generator(device="cuda:0").manual_seed(seed)


def _weights(t, nrows, k, gen):
    """random blocks whose dequantized values look like N(0, 0.02), in the device layout"""
    return mi355.upload_weights(t, lg.random_quantized(t, nrows, k, torch.device("cuda:0"), gen))


def _causal_mask(Nq, Nkv):
    """llama.cpp's mask: rows padded to 64, the last query sees every cell"""
    npad = (Nq + 63) // 64 * 64
    rows = torch.arange(npad, device="cuda:0")[:, None]
    cols = torch.arange(Nkv, device="cuda:0")[None, :]
    mask = torch.full((npad, Nkv), float("-inf"), dtype=torch.float16, device="cuda:0")
    mask[(cols <= Nkv - Nq + rows) & (rows < Nq)] = 0.0
    return mask


def _model(case, seed, T):
    cfg = lg.LlamaConfig(n_layer=case["layers"], n_embd=case["embd"], n_ff=case["ff"], n_head=case["H"], n_head_kv=case["HK"], n_vocab=case["vocab"], n_ctx=case["n_kv"])
    run = lg.LlamaRunner(lg.LlamaWeights(cfg, torch.device("cuda:0"), seed=seed, ftype=case["ftype"], quantize=True), max_tokens=T)
    gen = _gen(seed + 1)
    for c in run.kcache + run.vcache:      # what earlier tokens have left in the cache
        c.normal_(generator=gen)
    emb = torch.randn(T, case["embd"], device="cuda:0", generator=gen)
    return run, emb


def prepare(case, seed):
    kind = case["kind"]
    gen = _gen(seed)
    dev = torch.device("cuda:0")
    if kind == "mm":
        t = mi355.WEIGHT_TYPES[case["type"]]
        return {"kind": kind, "t": t, "W": _weights(t, case["N"], case["K"], gen), "x": torch.randn(case["B"], case["K"], device=dev, generator=gen)}
    if kind == "mmid":
        t = mi355.WEIGHT_TYPES[case["type"]]
        N, K, E, T = case["N"], case["K"], case["E"], case["T"]
        W = _weights(t, E * N, K, gen).reshape(E, N, -1)
        ids = torch.rand(T, E, device=dev, generator=gen).argsort(dim=1).to(torch.int32)[:, :case["used"]].contiguous()
        return {"kind": kind, "t": t, "W": W, "b": torch.randn(T, 1, K, device=dev, generator=gen), "ids": ids, "used": case["used"]}
    if kind == "fa":
        D, H, HK, Nq, Nkv = case["D"], case["H"], case["HK"], case["Nq"], case["Nkv"]
        q = torch.randn(Nq, H, D, device=dev, generator=gen).permute(1, 0, 2)
        k = torch.randn(Nkv, HK, D, device=dev, generator=gen).half().permute(1, 0, 2)
        v = torch.randn(Nkv, HK, D, device=dev, generator=gen).half().permute(1, 0, 2)
        return {"kind": kind, "q": q, "k": k, "v": v, "mask": _causal_mask(Nq, Nkv), "scale": 1.0 / math.sqrt(D)}
    if kind == "fa_kv":
        D, H, HK, Nkv = case["D"], case["H"], case["HK"], case["Nkv"]
        t = mi355.WEIGHT_TYPES[case["cache"]]
        lib = mi355.load()
        blocks = HK * D // 32                 # per cell; the whole cache is one row of the device row layout
        caches = []
        for _ in range(2):
            src = torch.randn(Nkv, HK * D, device=dev, generator=gen)
            c = torch.empty(Nkv * blocks * mi355.BLOCK[t][1], dtype=torch.uint8, device=dev)
            mi355.check(lib.mi355_cpy_f32_quant(torch.cuda.current_stream().cuda_stream, t, src.data_ptr(), c.data_ptr(), 0, Nkv * blocks, Nkv * HK * D))
            caches.append(c)
        need = int(lib.mi355_flash_attn_kv_ws_bytes(D, 1, Nkv, H, HK, t, t))
        return {"kind": kind, "t": t, "k": caches[0], "v": caches[1], "q": torch.randn(1, H, D, device=dev, generator=gen), "mask": _causal_mask(1, Nkv), "D": D, "H": H, "HK": HK,
                "Nkv": Nkv, "dst": torch.empty(1, H, D, device=dev), "ws": torch.empty(need + 256, dtype=torch.uint8, device=dev)}
    n_kv = case["n_kv"]
    if kind == "decode":
        run, emb = _model(case, seed, 1)
        run.pos.fill_(n_kv - 1)
        run.mask.fill_(float("-inf"))
        run.mask[0, :n_kv] = 0.0
        stream = torch.cuda.Stream()
        stream.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(stream):
            run.forward(1, n_kv)
            stream.synchronize()
            graph = torch.cuda.CUDAGraph()
            with torch.cuda.graph(graph, stream=stream):
                run.forward(1, n_kv)
        torch.cuda.synchronize()
        return {"kind": kind, "run": run, "emb": emb, "graph": graph}
    T = case["T"]
    run, emb = _model(case, seed, T)
    run.set_inputs(emb, n_kv - T, T, n_kv)
    run.forward(T, n_kv)                      # lays the weights out for prompt batches, once per model
    return {"kind": kind, "run": run, "emb": emb, "T": T, "n_kv": n_kv}


# ---------------------------------------------------------------------------------------------- one pass
def run(state):
    kind = state["kind"]
    if kind == "mm":
        return mi355.mul_mat(state["t"], state["W"], state["x"])
    if kind == "mmid":
        return mi355.mul_mat_id(state["t"], state["W"], state["b"], state["ids"], state["used"])
    if kind == "fa":
        return mi355.flash_attn_ext(state["q"], state["k"], state["v"], state["mask"], state["scale"])
    if kind == "fa_kv":
        D, H, HK, Nkv, t = state["D"], state["H"], state["HK"], state["Nkv"], state["t"]
        bb = mi355.BLOCK[t][1]
        head, cell = D // 32 * bb, HK * D // 32 * bb
        k, v, ws = state["k"].data_ptr(), state["v"].data_ptr(), (state["ws"].data_ptr() + 255) & ~255
        blocks = Nkv * HK * D // 32
        mi355.check(mi355.load().mi355_flash_attn_ext_kv(torch.cuda.current_stream().cuda_stream, state["q"].data_ptr(), k, t, k, blocks, v, t, v, blocks, state["mask"].data_ptr(),
                                                         state["dst"].data_ptr(), D, 1, Nkv, H, HK, H * D * 4, D * 4, cell, head, cell, head, state["mask"].stride(0) * 2,
                                                         1.0 / math.sqrt(D), 0.0, 0.0, ws, state["ws"].numel() - 256, None))
        return state["dst"]
    r = state["run"]
    if kind == "decode":
        r.x[:1].copy_(state["emb"])
        state["graph"].replay()
        return {"logits": r.logits[:1], "hidden": r.x[:1], "k": r.kcache[-1], "v": r.vcache[-1]}
    T = state["T"]
    r.x[:T].copy_(state["emb"])
    logits = r.forward(T, state["n_kv"])
    return {"logits": logits, "hidden": r.x[:T], "k": r.kcache[-1], "v": r.vcache[-1]}


# ---------------------------------------------------------------------------------------------- what a pass cannot do without
def _wbytes(t, n, k):
    be, bb = mi355.BLOCK[mi355.WEIGHT_TYPES[t]]
    return n * (k // be) * bb


def work(case):
    kind = case["kind"]
    if kind == "mm":
        N, K, B = case["N"], case["K"], case["B"]
        return {"bytes": _wbytes(case["type"], N, K) + 4 * B * (K + N), "flops": 2 * N * K * B}
    if kind == "mmid":
        N, K, E, T, u = case["N"], case["K"], case["E"], case["T"], case["used"]
        touched = E * (1.0 - (1.0 - u / E) ** T)           # experts that any token uses, on average
        return {"bytes": touched * _wbytes(case["type"], N, K) + 4 * T * K + 4 * T * u * N + 4 * T * u, "flops": 2 * N * K * T * u}
    if kind in ("fa", "fa_kv"):
        D, H, HK, Nq, Nkv = case["D"], case["H"], case["HK"], case.get("Nq", 1), case["Nkv"]
        pairs = Nq * (Nkv - Nq) + Nq * (Nq + 1) // 2       # visible (query, cell) pairs of the causal mask
        cell = {"fa": 2.0, "fa_kv": 34 / 32 if case.get("cache") == "q8_0" else 18 / 32}[kind]
        return {"bytes": 2 * cell * HK * D * Nkv + 8 * Nq * H * D + 2 * Nq * Nkv, "flops": 4 * H * D * pairs}
    L, E, F, D, V = case["layers"], case["embd"], case["ff"], 128, case["vocab"]
    qd, kd = case["H"] * D, case["HK"] * D
    base = {"q4_k_m": "q4_K", "q8_0": "q8_0", "q4_0": "q4_0"}[case["ftype"]]
    total = 0
    for il in range(L):
        vt = "q6_K" if case["ftype"] == "q4_k_m" and lg.use_more_bits(il, L) else base
        total += _wbytes(base, qd, E) + _wbytes(base, kd, E) + _wbytes(vt, kd, E) + _wbytes(base, E, qd) + 2 * _wbytes(base, F, E) + _wbytes(vt, E, F)
    total += _wbytes("q6_K" if case["ftype"] == "q4_k_m" else base, V, E)
    T, n_kv = case.get("T", 1), case["n_kv"]
    total += L * 2 * 2 * kd * n_kv + 8 * T * E + 4 * V
    params = L * (2 * qd * E + 2 * kd * E + 3 * F * E)
    pairs = T * (n_kv - T) + T * (T + 1) // 2
    return {"bytes": total, "flops": 2 * params * T + 2 * V * E + 4 * L * qd * pairs}


def tolerance(case):
    """Four times (rounded) what the same path differs from 64-bit arithmetic on the same quantized operands - for whole models, from
    itself when the embedding moves by half a unit in the last place."""
    kind = case["kind"]
    if kind in ("mm", "mmid"):
        rows = case["B"] if kind == "mm" else case["T"] * case["used"]
        if case["type"] in ("q4_1", "q5_1") and rows >= 32:
            return {"rel": 1.5e-3}    # block_q8_1 carries scale * sum as f16: 3.7e-4
        return {"rel": 1e-6}          # exact integer dots of a block, f32 sums over the blocks: 7e-8 .. 1.6e-7
    if kind == "fa":
        return {"rel": 1.2e-3}        # f16 cache and probabilities: 2e-4 .. 3e-4
    if kind == "fa_kv":
        return {"rel": 2e-2}          # the query is quantized to the cache's 8-bit blocks: 5e-3
    # activations are quantized to 8 bits before every product: a sum that rounds the other way moves a level by 1/127 of its block's
    # maximum, and from there on every later level is drawn anew.  0.03 .. 0.05 at 8 layers, 0.07 .. 0.11 at 32
    return {"rel": 0.08 * math.sqrt(case["layers"])}
