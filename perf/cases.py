"""The attention work an engine has this library do, as cases that can be timed and compared: one pass each through the
public entry points (nextsycl_amd.attn.Ops), inputs resident on the GPU.

Four kinds of pass ("op"):
  gqa   grouped-query attention over a KV cache: up to 16 rows are a decode or verify pass (ns_attn_decode_t), more a
        prompt pass (ns_attn_prompt_t). "store": the pass begins as a layer's does, with its rows' q / k norm, rotary
        positions and cache rows (ns_attn_pre_store). "window": a sliding window over a ring cache.
  mla   absorbed multi-head latent attention: "full" a token from its projections to the value up-projection
        (ns_ds2_kv_store, ns_ds2_mla_decode), else rows already absorbed (ns_mla_decode_latent).
  mm3   block-sparse attention of a position-major cache: block scores, the best blocks a (row, key head), attention over
        them (ns_llm_minimaxm3_idx_scores / _idx_topk / _attend).
  glm   latent attention over selected pools of 4 cells: the row's own latent cells and pooled keys, the pool scores, the
        best pools a row, attention over them (ns_to_q8row or ns_to_f16, ns_idx_pool, ns_gemm_f16, ns_idx_score, ns_topk,
        ns_mla_attend_sel(_q8))."""
import math

import torch

from nextsycl_amd import DevBuf, Gpu
from nextsycl_amd.attn import BF16, ELT, F16, F32, KV_BF16, KV_F16, KV_Q4_0, KV_Q8_0, Ops, kv_row_bytes

IO = {"f32": (F32, torch.float32), "f16": (F16, torch.float16), "bf16": (BF16, torch.bfloat16)}
CACHE = {"f16": (KV_F16, torch.float16), "q8_0": (KV_Q8_0, torch.uint8), "q4_0": (KV_Q4_0, torch.uint8), "bf16": (KV_BF16, torch.bfloat16)}
LATENT, ROPE = 512, 64            # an MLA cell: latent features, rotated key features
IDX_HEADS, IDX_DIM = 32, 128      # the pool indexer's query heads and key width
MM3_D, MM3_BLOCK = 128, 128       # block-sparse: head size, keys a block
EPS, THETA = 1e-6, 1e6


def listed():
    return [
        # a token of a short chat, one layer: the smallest pass an engine makes, three short launches
        {"name": "token_1k", "op": "gqa", "rows": 1, "heads": 32, "kv_heads": 8, "head": 128, "cache": "f16", "io": "f16", "past": 999, "window": 0,
         "store": True},
        # a token behind a long context in half precision
        {"name": "decode_32k", "op": "gqa", "rows": 1, "heads": 32, "kv_heads": 8, "head": 128, "cache": "f16", "io": "f16", "past": 32767, "window": 0,
         "store": False},
        # a token behind a very long context, the cache quantized to hold it
        {"name": "decode_128k_q8", "op": "gqa", "rows": 1, "heads": 64, "kv_heads": 4, "head": 128, "cache": "q8_0", "io": "f16", "past": 131071,
         "window": 0, "store": False},
        # a speculative verify pass of four rows over heads of 256 and the smallest cache form, one layer
        {"name": "verify_43k_q4", "op": "gqa", "rows": 4, "heads": 24, "kv_heads": 4, "head": 256, "cache": "q4_0", "io": "f32", "past": 43003, "window": 0,
         "store": True},
        # a whole prompt at once, bfloat16 throughout
        {"name": "prompt_8k", "op": "gqa", "rows": 8192, "heads": 40, "kv_heads": 8, "head": 128, "cache": "bf16", "io": "bf16", "past": 0, "window": 0,
         "store": False},
        # a chunk in the middle of a prompt, heads of 256 over a quantized cache, one layer
        {"name": "prompt_chunk_q8", "op": "gqa", "rows": 2048, "heads": 24, "kv_heads": 4, "head": 256, "cache": "q8_0", "io": "f32", "past": 8192,
         "window": 0, "store": True},
        # a ragged chunk through a sliding-window layer's ring cache
        {"name": "prompt_window", "op": "gqa", "rows": 2001, "heads": 32, "kv_heads": 2, "head": 128, "cache": "f16", "io": "f32", "past": 10007,
         "window": 1024, "store": False},
        # a short follow-up question behind the conversation so far, one layer
        {"name": "new_turn", "op": "gqa", "rows": 37, "heads": 32, "kv_heads": 8, "head": 128, "cache": "bf16", "io": "bf16", "past": 20011, "window": 0,
         "store": True},
        # a token of a latent-attention model, from its projections to the heads' values
        {"name": "mla_token", "op": "mla", "rows": 1, "heads": 128, "past": 32767, "io": "f32", "full": True},
        # a prompt chunk of the same model
        {"name": "mla_prompt", "op": "mla", "rows": 256, "heads": 128, "past": 8192, "io": "f16", "full": False},
        # a prompt chunk through a block-sparse layer, its indexer included
        {"name": "sparse_prompt", "op": "mm3", "rows": 1024, "heads": 64, "kv_heads": 4, "past": 16384, "blocks": 16},
        # two rows (a token and its draft) through a pool-sparse latent layer, its indexer included
        {"name": "sparse_token", "op": "glm", "rows": 2, "heads": 64, "past": 100001, "cache": "q8_0", "pools": 512},
    ]


def _log(rng, lo, hi):
    """A whole number between lo and hi, spread over its logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


# (query heads, key heads, head size) of this library's engines and workloads
HEADS = [(32, 8, 128), (40, 8, 128), (64, 4, 128), (32, 4, 128), (32, 2, 128), (16, 4, 128), (24, 4, 256), (16, 2, 256), (12, 2, 256)]
# no drawn pass asks for more than the largest listed ones
MOST_FLOPS, MOST_BYTES = 5.0e11, 1.4e8


def draw(rng):
    kind = rng.choice(["decode", "decode", "verify", "prompt", "prompt", "turn", "window", "mla_token", "mla_prompt", "mm3", "mm3_token", "glm"])
    if kind in ("decode", "verify", "prompt", "turn", "window"):
        Hq, Hkv, D = rng.choice(HEADS)
        cache = rng.choice(["f16", "bf16"] if kind == "window" else ["f16", "q8_0", "q4_0", "bf16"])
        io = "bf16" if cache == "bf16" else rng.choice(["f32", "f16"])
        rows = {"decode": 1, "verify": rng.randint(2, 8), "turn": _log(rng, 17, 128)}.get(kind) or _log(rng, 129, 8192)
        past = _log(rng, 250, 131071)
        if kind in ("prompt", "window"):
            past = rng.choice([0, _log(rng, 250, 32768)])
        window = _log(rng, 128, 4096) if kind == "window" else 0
        case = {"op": "gqa", "rows": rows, "heads": Hq, "kv_heads": Hkv, "head": D, "cache": cache, "io": io, "past": past, "window": window,
                "store": rng.random() < 0.5}
        while True:
            w = work(case)
            if w["flops"] <= MOST_FLOPS and w["bytes"] - 8 * case["rows"] * Hq * D <= MOST_BYTES:
                return case
            if case["past"] > 250:
                case["past"] = int(case["past"] * 0.8)
            else:
                case["rows"] = int(case["rows"] * 0.9)
    if kind == "mla_token":
        return {"op": "mla", "rows": rng.randint(1, 4), "heads": rng.choice([16, 64, 128]), "past": _log(rng, 250, 65536), "io": "f32", "full": True}
    if kind == "mla_prompt":
        heads, rows = rng.choice([16, 64, 128]), _log(rng, 17, 512)
        return {"op": "mla", "rows": rows, "heads": heads, "past": min(_log(rng, 250, 32768), 256 * 128 * 8192 // (rows * heads)), "io": rng.choice(["f32", "f16"]),
                "full": False}
    if kind in ("mm3", "mm3_token"):
        rows = rng.randint(1, 4) if kind == "mm3_token" else _log(rng, 17, 1024)
        most = 131072 if kind == "mm3_token" else min(65536, 1024 * 16384 // rows)
        return {"op": "mm3", "rows": rows, "heads": 64, "kv_heads": 4, "past": _log(rng, 3000, most), "blocks": 16}
    rows = rng.choice([rng.randint(1, 8), _log(rng, 17, 128)])
    return {"op": "glm", "rows": rows, "heads": 64, "past": _log(rng, 9000, 131072 if rows <= 8 else 65536), "cache": rng.choice(["f16", "q8_0"]), "pools": 512}


# ---- what a program has in hand before the call

_ops = []


def _engine():
    """The one GPU handle a program opens."""
    if not _ops:
        _ops.append(Ops(Gpu.open(0)))
    return _ops[0]


def _buf(t):
    """A tensor's memory as the library's buffer."""
    return DevBuf(_engine().gpu, t.numel() * t.element_size(), _ptr=t.data_ptr(), _owner=t)


class _Random:
    def __init__(self, seed):
        self.g = torch.Generator("cuda").manual_seed(seed)

    def __call__(self, *shape, sigma=1.0, dtype=torch.float32):
        return (torch.randn(*shape, generator=self.g, device="cuda") * sigma).to(dtype)


def _settled():
    """Torch's stream and the library's are two: what one has written, the other may read after this."""
    torch.cuda.synchronize()


def prepare(case, seed):
    state = {"gqa": _prepare_gqa, "mla": _prepare_mla, "mm3": _prepare_mm3, "glm": _prepare_glm}[case["op"]](case, _Random(seed))
    state["case"] = case
    _settled()
    return state


def _prepare_gqa(c, rand):
    ops = _engine()
    T, Hq, Hkv, D, p0 = c["rows"], c["heads"], c["kv_heads"], c["head"], c["past"]
    kt, ktype = CACHE[c["cache"]]
    qt, qtype = IO[c["io"]]
    n = p0 + T
    ring = c["window"] > 0
    cap = min(n, c["window"] + T) if ring else n
    row = kv_row_bytes(kt, D) // (1 if ktype is torch.uint8 else 2)
    s = {"kc": torch.zeros(Hkv, cap, row, dtype=ktype, device="cuda"), "vc": torch.zeros(Hkv, cap, row, dtype=ktype, device="cuda"), "cap": cap}
    # the context's rows, stored a chunk at a time; the pass's own too unless it stores them itself
    end, at = (p0 if c["store"] else n), max(0, n - cap)
    kc, vc = _buf(s["kc"]), _buf(s["vc"])
    while at < end:
        m = min(16384, cap, end - at)
        k, v = rand(m, Hkv * D), rand(m, Hkv * D)
        _settled()
        ops.kv_store(kt, _buf(k), Hkv * D, _buf(v), Hkv * D, m, Hkv, D, cap, at, kc, vc, ring=ring)
        _settled()
        at += m
    s["q"] = torch.empty(T, Hq * D, dtype=qtype, device="cuda") if c["store"] else rand(T, Hq * D, dtype=qtype)
    s["out"] = torch.empty(T, Hq, D, dtype=qtype, device="cuda")
    s["b"] = {"kc": kc, "vc": vc, "q": _buf(s["q"]), "out": _buf(s["out"])}
    if c["store"]:
        s["raw"] = [rand(T, h * D) for h in (Hq, Hkv, Hkv)] + [1.0 + 0.1 * rand(D) for _ in range(2)]
        s["b"]["raw"] = [_buf(t) for t in s["raw"]]
    s["scratch"] = DevBuf(ops.gpu, max(4, 4 * ops.decode_scratch(T, Hq, Hkv, D, p0, c["window"]))) if T <= 16 else None
    return s


def _run_gqa(c, s):
    ops, b = _engine(), s["b"]
    T, Hq, Hkv, D, p0, win, cap = c["rows"], c["heads"], c["kv_heads"], c["head"], c["past"], c["window"], s["cap"]
    kt, qt = CACHE[c["cache"]][0], IO[c["io"]][0]
    if c["store"]:
        q, k, v, qw, kw = b["raw"]
        ops.pre_store(1, qt, kt, win > 0, q, Hq * D, D, b["q"], Hq * D, k, Hkv * D, D, v, Hkv * D, qw, kw, EPS, D // 2, THETA, T, Hq, Hkv, D, cap, p0,
                      b["kc"], b["vc"])
    if T <= 16:
        ops.decode(qt, kt, b["q"], Hq * D, b["kc"], b["vc"], T, Hq, Hkv, D, cap, p0, b["out"], s["scratch"], win=win)
    else:
        ops.prompt(qt, kt, b["q"], Hq * D, b["kc"], b["vc"], T, Hq, Hkv, D, cap, p0, b["out"], win=win)
    return {"out": s["out"], "kc": s["kc"], "vc": s["vc"]} if c["store"] else s["out"]


def _prepare_mla(c, rand):
    ops = _engine()
    T, H, p0 = c["rows"], c["heads"], c["past"]
    s = {"cache": rand(p0 + T, LATENT + ROPE, sigma=0.5, dtype=torch.float16)}
    if c["full"]:
        s["kv"], s["w"] = rand(T, LATENT + ROPE), 0.5 + 0.05 * rand(LATENT)
        # (projections of the size that leaves absorbed queries and values of order one)
        s["q"], s["kb"], s["vb"] = rand(T, H, 192), rand(H, LATENT, 128, sigma=128 ** -0.5, dtype=torch.float16), rand(H, 128, LATENT, sigma=LATENT ** -0.5, dtype=torch.float16)
        s["out"] = torch.empty(T, H, 128, device="cuda")
    else:
        qtype = IO[c["io"]][1]
        s["q"], s["out"] = rand(T, H, LATENT + ROPE, dtype=qtype), torch.empty(T, H, LATENT, dtype=qtype, device="cuda")
    s["b"] = {k: _buf(t) for k, t in s.items()}
    if not c["full"]:
        s["scratch"] = DevBuf(ops.gpu, max(4, 4 * ops.mla_latent_scratch(T, H, p0)))
    return s


def _run_mla(c, s):
    ops, b = _engine(), s["b"]
    T, H, p0 = c["rows"], c["heads"], c["past"]
    if not c["full"]:
        ops.mla_decode_latent(IO[c["io"]][0], b["q"], b["cache"], b["out"], T, H, ROPE, p0, 192.0 ** -0.5, s["scratch"])
        return s["out"]
    ops.ds2_kv_store(b["kv"], b["w"], EPS, b["cache"], T, LATENT, ROPE, p0, 10000.0, 1.0, 0.0, 1.0, 0.0, 0.0)
    ops.mla_decode(b["q"], b["kb"], b["vb"], b["cache"], b["out"], T, H, p0, 192.0 ** -0.5)
    return {"out": s["out"], "cells": s["cache"][p0:]}


def _prepare_mm3(c, rand):
    T, Hq, Hkv, p0, K = c["rows"], c["heads"], c["kv_heads"], c["past"], c["blocks"]
    n = p0 + T
    nblk = (n + MM3_BLOCK - 1) // MM3_BLOCK
    s = {"kc": rand(n, Hkv, MM3_D, dtype=torch.float16), "vc": rand(n, Hkv, MM3_D, dtype=torch.float16), "q": rand(T, Hq, MM3_D),
         "iq": rand(T, Hkv, MM3_D), "ik": rand(n, MM3_D, dtype=torch.float16), "scores": torch.empty(T, Hkv, nblk, device="cuda"),
         "sel": torch.empty(T, Hkv, K, dtype=torch.int32, device="cuda"), "out": torch.empty(T, Hq, MM3_D, device="cuda")}
    s["b"] = {k: _buf(t) for k, t in s.items()}
    s["nblk"] = nblk
    return s


def _run_mm3(c, s):
    ops, b = _engine(), s["b"]
    T, Hq, Hkv, p0, K = c["rows"], c["heads"], c["kv_heads"], c["past"], c["blocks"]
    ops.minimaxm3_idx_scores(b["iq"], b["ik"], b["scores"], T, Hkv, s["nblk"], p0, 1)
    ops.minimaxm3_idx_topk(b["scores"], b["sel"], T, Hkv, s["nblk"], K)
    ops.minimaxm3_attend(b["q"], b["kc"], b["vc"], b["out"], T, Hq, Hkv, p0, MM3_D ** -0.5, sel=b["sel"], K=K)
    return {"out": s["out"], "sel": s["sel"]}


def _prepare_glm(c, rand):
    T, H, p0, K = c["rows"], c["heads"], c["past"], c["pools"]
    n, npool = p0 + T, (p0 + T) // 4
    q8 = c["cache"] == "q8_0"
    s = {"x": rand(n, LATENT), "cells": torch.zeros(n, LATENT // 32 * 2 + LATENT, dtype=torch.uint8, device="cuda") if q8 else
         torch.zeros(n, LATENT, dtype=torch.float16, device="cuda")}
    ops = _engine()
    _settled()
    _store_cells(ops, q8, _buf(s["x"]), _buf(s["cells"]), n)
    _settled()
    s["x"] = s["x"][p0:].clone()                      # the pass's own rows, stored again by the pass
    s.update({"own": s["cells"][p0:], "qa": rand(T, H, LATENT, sigma=0.3), "u": torch.empty(T, H, LATENT, device="cuda"),
              "iq": rand(T, IDX_HEADS, IDX_DIM, dtype=torch.float16), "w": rand(T, IDX_HEADS), "ik": rand(T, IDX_DIM), "ig": rand(T, IDX_DIM),
              "ape": rand(4, IDX_DIM, sigma=0.5), "ring": rand(8, 2 * IDX_DIM), "pooled": rand(npool, IDX_DIM),
              "S": torch.empty(T * IDX_HEADS, npool, device="cuda"), "score": torch.empty(T, npool, device="cuda"),
              "sel": torch.zeros(T, K, dtype=torch.int32, device="cuda"), "cnt": torch.full((T,), K, dtype=torch.int32, device="cuda")})
    s["pooled_h"] = s["pooled"].to(torch.float16)
    s["b"] = {k: _buf(t) for k, t in s.items()}
    # the pools this pass completes, as the half rows the scores' product reads
    j0 = p0 // 4
    s["new"] = (s["b"]["pooled"].view(j0 * IDX_DIM * 4, (npool - j0) * IDX_DIM * 4), s["b"]["pooled_h"].view(j0 * IDX_DIM * 2, (npool - j0) * IDX_DIM * 2),
                (npool - j0) * IDX_DIM)
    return s


def _store_cells(ops, q8, x, cells, n):
    if q8:
        ops.to_q8row(x, cells, n, LATENT)
    else:
        ops.to_f16(x, cells, n * LATENT)


def _run_glm(c, s):
    ops, b = _engine(), s["b"]
    T, H, p0, K = c["rows"], c["heads"], c["past"], c["pools"]
    npool, q8 = (p0 + T) // 4, c["cache"] == "q8_0"
    _store_cells(ops, q8, b["x"], b["own"], T)
    ops.ok(ops.k.idx_pool(ops.raw(), b["ring"].ptr, b["ik"].ptr, b["ig"].ptr, b["ape"].ptr, b["pooled"].ptr, p0, T, IDX_DIM), "idx_pool")
    pooled, pooled_h, fresh = s["new"]
    if fresh:
        ops.to_f16(pooled, pooled_h, fresh)
    ops.gemm_f16(T * IDX_HEADS, npool, IDX_DIM, b["iq"], IDX_DIM, b["pooled_h"], b["S"], npool)
    ops.ok(ops.k.idx_score(ops.raw(), b["S"].ptr, b["w"].ptr, b["score"].ptr, T, IDX_HEADS, 0, npool, npool, p0), "idx_score")
    ops.ok(ops.k.topk(ops.raw(), b["score"].ptr, b["sel"].ptr, T, npool, npool, K), "topk")
    ops.mla_attend(b["qa"], b["cells"], b["u"], T, H, LATENT, p0, 192.0 ** -0.5, q8=q8, sel=b["sel"], sel_cnt=b["cnt"], K=K)
    # (the lists and scores live from the indexer to the attention of the same layer: what leaves it is u, and the rows
    # the pass has added)
    return {"u": s["u"], "own": s["own"], "ring": s["ring"], "pooled": s["pooled"]}


def run(state):
    return {"gqa": _run_gqa, "mla": _run_mla, "mm3": _run_mm3, "glm": _run_glm}[state["case"]["op"]](state["case"], state)


# ---- what a pass cannot do without, and how close two right answers are

def work(case):
    c, T, p0 = case, case["rows"], case["past"]
    n = p0 + T
    pairs = T * p0 + T * (T + 1) // 2                                  # (row, key it sees)
    if c["op"] == "gqa":
        Hq, Hkv, D, win = c["heads"], c["kv_heads"], c["head"], c["window"]
        keys = n
        if win:
            keys = min(n, win + T - 1)
            pairs = sum(min(win, p0 + t + 1) for t in range(T))
        e = ELT[IO[c["io"]][0]]
        nbytes = 2 * Hkv * keys * kv_row_bytes(CACHE[c["cache"]][0], D) + T * Hq * D * ((4 if c["store"] else e) + e) + (8 * T * Hkv * D if c["store"] else 0)
        return {"bytes": nbytes, "flops": 4 * pairs * Hq * D}
    if c["op"] == "mla":
        H, e = c["heads"], ELT[IO[c["io"]][0]]
        flops, nbytes = 2 * pairs * H * (2 * LATENT + ROPE), n * (LATENT + ROPE) * 2
        if c["full"]:
            return {"bytes": nbytes + H * 2 * 128 * LATENT * 2 + T * H * (192 + 128) * 4 + T * (LATENT + ROPE) * 4, "flops": flops + T * H * 4 * 128 * LATENT}
        return {"bytes": nbytes + T * H * (2 * LATENT + ROPE) * e, "flops": flops}
    if c["op"] == "mm3":
        Hq, Hkv, seen = c["heads"], c["kv_heads"], c["blocks"] * MM3_BLOCK
        nbytes = n * MM3_D * 2 + 2 * Hkv * min(n, T * seen) * MM3_D * 2 + T * (2 * Hq + Hkv) * MM3_D * 4
        return {"bytes": nbytes, "flops": 2 * pairs * Hkv * MM3_D + 4 * T * Hq * MM3_D * seen}
    H, cells, cell = c["heads"], 4 * c["pools"], LATENT // 32 * 2 + LATENT if c["cache"] == "q8_0" else 2 * LATENT
    nbytes = n // 4 * IDX_DIM * 2 + min(n, T * cells) * cell + 2 * T * H * LATENT * 4 + T * LATENT * 4
    return {"bytes": nbytes, "flops": 2 * T * IDX_HEADS * (n // 4) * IDX_DIM + 4 * T * H * cells * LATENT}


def tolerance(case):
    """Softmax weights, and keys and values where a cache is wider or narrower than the matrix unit's operands, enter the
    products rounded to half; rows leave in their own type. Against float64 the passes sit at 2.2e-4 .. 4.1e-4 (largest
    difference 7e-4 .. 1.7e-3) with float32 or half rows, at 1.1e-3 .. 1.7e-3 (4.1e-3) with bfloat16 ones."""
    rel, most = {"f32": (1.6e-3, 0.01), "f16": (1.6e-3, 0.01), "bf16": (6.6e-3, 0.03)}[case.get("io", "f32")]
    if case["op"] == "mm3":
        # two blocks whose scores agree to the last bits may change places in a list, or one may stand for the other at its
        # end: another block of sixteen for one (row, key head)
        return {"rel": 1e-2, "max": 0.9, "differ": 1e-3}
    return {"rel": rel, "max": most}
