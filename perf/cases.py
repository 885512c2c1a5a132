"""The work a host engine gives this library, as timing cases.

Each case goes through the public C entry points the way an engine calls
them:

  gemv     q4_mmvq_n over `mats` weight matrices, one after another
           (projections of successive layers, or one LM head); with graph the
           calls are captured once and replayed, as a decode step is
  decode   one token through `layers` routed-expert layers: host lists
           (q4_hip_moe_exec) or, routed, the router and the layer together
           (q4mi_moe_route_exec); captured once, replayed per token
  window   a verify window of 2..8 tokens through `layers` layers
           (q4_hip_moe_exec_win over device lists), captured
  prefill  one routed layer over a prompt: route, pack, q8(x), gate/up, down,
           weighted reduce, with the shared expert in the same launches
  xg       the fp16-activation prefill of the same layer over a tile table

Weights are random blocks of the named format (every index, sign and
sub-block scale uniform) whose block scales give weights of about 0.025 rms;
activations are N(0,1); every layer of a stack has its own weights, so a pass
streams them from HBM.  Routing follows router logits N(0,1), with a Zipf
popularity bias for prompts.
"""
import ctypes
import math
import os
import re
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "suzuku-engine-q4_amd"))
import q4mi  # noqa: E402

# format: (type id, values per block, bytes per block, offset of the fp16
# scale, block scale for weights of about 0.025 rms)
FORMATS = {
    "Q8_0": (8, 32, 34, 0, 3.4e-4),
    "Q6_K": (14, 256, 210, 208, 1.8e-5),
    "IQ3_XXS": (18, 256, 98, 0, 1.5e-4),
    "IQ4_NL": (20, 32, 18, 0, 3.7e-4),
    "IQ3_S": (21, 256, 110, 0, 1.7e-4),
    "IQ2_S": (22, 256, 82, 0, 3.9e-4),
    "IQ4_XS": (23, 256, 136, 0, 2.0e-5),
    "Q2_0": (42, 64, 18, 0, 2.0e-2),
}
SHARED = 1          # shared experts beside the routed ones


def listed():
    return [
        # the smallest call of a decode step: one short projection, alone
        {"name": "gemv_small", "kind": "gemv", "type": "IQ3_S", "rows": 1024, "cols": 2048,
         "n": 1, "mats": 1, "graph": False},
        # square IQ3_S projections of successive layers in a decode step
        {"name": "gemv_iq3s", "kind": "gemv", "type": "IQ3_S", "rows": 4096, "cols": 4096,
         "n": 1, "mats": 24, "graph": True},
        # the LM head of a decode step, one token
        {"name": "lm_head_1", "kind": "gemv", "type": "Q8_0", "rows": 151936, "cols": 2048,
         "n": 1, "mats": 1, "graph": False},
        # the LM head of a verify window, four tokens
        {"name": "lm_head_4", "kind": "gemv", "type": "Q8_0", "rows": 151936, "cols": 2048,
         "n": 4, "mats": 1, "graph": False},
        # one token through a stack of routed layers, lists from the host
        {"name": "decode", "kind": "decode", "routed": False, "gate": "IQ3_S", "down": "IQ3_S",
         "hidden": 2048, "ff": 512, "experts": 64, "topk": 10, "layers": 24},
        # the same with the router on the device ahead of every layer
        {"name": "decode_routed", "kind": "decode", "routed": True, "gate": "IQ3_S",
         "down": "IQ3_S", "hidden": 2048, "ff": 512, "experts": 512, "topk": 10, "layers": 12},
        # a four-token verify window (one accepted, three drafted)
        {"name": "window_4", "kind": "window", "gate": "IQ3_S", "down": "IQ3_S", "hidden": 2048,
         "ff": 512, "experts": 512, "topk": 10, "tokens": 4, "layers": 8},
        # the reference model's mixed-format window at its own sizes
        {"name": "window_mixed", "kind": "window", "gate": "IQ2_S", "down": "IQ4_NL",
         "hidden": 2560, "ff": 640, "experts": 256, "topk": 10, "tokens": 4, "layers": 8},
        # a whole prompt chunk through one layer
        {"name": "prefill_2048", "kind": "prefill", "gate": "IQ3_S", "down": "IQ3_S",
         "hidden": 2048, "ff": 512, "experts": 512, "topk": 10, "tokens": 2048},
        # a short ragged prompt: most experts get a handful of rows
        {"name": "prefill_333", "kind": "prefill", "gate": "IQ3_S", "down": "IQ3_S",
         "hidden": 2048, "ff": 512, "experts": 512, "topk": 10, "tokens": 333},
        # the mixed-format fp16-activation prefill
        {"name": "xg_1024", "kind": "xg", "gate": "IQ2_S", "down": "IQ4_NL", "hidden": 2048,
         "ff": 512, "experts": 256, "topk": 10, "tokens": 1024},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _draw(rng):
    kind = rng.choice(["gemv", "gemv", "decode", "window", "window", "prefill", "prefill", "xg"])
    if kind == "gemv":
        ty = rng.choice(["IQ3_S", "Q8_0", "IQ4_NL", "Q2_0", "IQ2_S", "Q6_K"])
        return {"kind": kind, "type": ty, "rows": _log(rng, 500, 160000),
                "cols": rng.choice([1024, 2048, 2560, 4096]), "n": rng.randint(1, 8),
                "mats": 1 if rng.random() < 0.7 else rng.randint(2, 12),
                "graph": rng.random() < 0.5}
    gate = rng.choice(["IQ3_S", "IQ3_S", "Q8_0", "IQ2_S"] +
                      ([] if kind in ("prefill", "xg") else ["IQ3_XXS", "IQ4_XS"]))
    down = rng.choice(["IQ3_S", "IQ3_S", "Q8_0", "IQ4_NL", "Q2_0"])
    ffs = [512, 1024] if down == "IQ3_S" or kind == "xg" else \
        [256, 512, 1024] if kind == "prefill" else [256, 512, 640, 1024]
    c = {"kind": kind, "gate": gate, "down": down, "ff": rng.choice(ffs),
         "hidden": rng.choice([1024, 2048, 2560, 4096]), "experts": rng.randint(16, 256),
         "topk": rng.randint(2, 10)}
    if kind == "decode":
        c.update(routed=rng.random() < 0.5, layers=rng.randint(1, 12))
    elif kind == "window":
        c.update(tokens=rng.randint(2, 8), layers=rng.randint(1, 8))
        c["topk"] = min(c["topk"], 64 // c["tokens"] - SHARED)
    else:
        c["tokens"] = _log(rng, 20, 2048)
    return c


def _cost(case):
    w = work(case)
    return w["bytes"] / 2e12 + w["flops"] / 2e14


def draw(rng):
    most = max(_cost(c) for c in listed())
    while True:
        c = _draw(rng)
        if _cost(c) <= most:
            return c


# ------------------------------------------------------------------ sizes

def _row_bytes(fmt, n):
    _, vals, size, _, _ = FORMATS[fmt]
    return n // vals * size


def _expert(case):
    """Bytes of one packed expert and the offsets of its up and down parts."""
    g = case["ff"] * _row_bytes(case["gate"], case["hidden"])
    d = case["hidden"] * _row_bytes(case["down"], case["ff"])
    return 2 * g + d, g, 2 * g


def _touched(case, tokens):
    """Expected number of routed experts that some token picks."""
    e, k = case["experts"], case["topk"]
    if case["kind"] not in ("prefill", "xg"):
        return e * (1.0 - (1.0 - k / e) ** tokens)
    ids = _zipf_logits(np.random.default_rng(1), tokens, e)
    return len(np.unique(np.argpartition(-ids, k - 1, axis=1)[:, :k]))


def work(case):
    if case["kind"] == "gemv":
        m, n = case["mats"], case["n"]
        rows, cols = case["rows"], case["cols"]
        return {"bytes": m * (rows * _row_bytes(case["type"], cols) + 4 * n * (rows + cols)),
                "flops": 2.0 * m * n * rows * cols}
    tokens, layers = case.get("tokens", 1), case.get("layers", 1)
    h, f = case["hidden"], case["ff"]
    weights = (_touched(case, tokens) + SHARED) * _expert(case)[0]
    routing = 4 * case["experts"] * (h + tokens) if case.get("routed") else 0
    rows = tokens * (case["topk"] + SHARED)
    return {"bytes": layers * (weights + routing + 8.0 * tokens * h),
            "flops": layers * (6.0 * rows * h * f + routing / 2.0)}


def tolerance(case):
    # Against 64 bits the GEMV differs by its fp32 sums of exact group sums.
    if case["kind"] == "gemv":
        return {"rel": 1e-6, "max": 1e-5}
    # A layer requantizes h = silu(gate) up between its two products: an h
    # within a few ulp of a rounding boundary takes the neighbouring q8 code
    # when its fp32 sums run in another order, which moves that expert's
    # output by up to 1/254 of the group's largest value.
    if case["kind"] == "xg":     # fp16 h: a rounding boundary every 2^-11
        return {"rel": 1e-4, "max": 2e-3, "differ": 1e-3}
    return {"rel": 4e-4, "max": 8e-3, "differ": 1e-3}


# ----------------------------------------------------------------- inputs

def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _blocks(fmt, count, gen):
    """Random blocks of a format, [count][bytes per block]."""
    _, _, size, at, scale = FORMATS[fmt]
    b = torch.randint(0, 256, (count, size), dtype=torch.uint8, device="cuda", generator=gen)
    if fmt == "Q8_0":      # codes -127..127
        q = b[:, 2:]
        q[q == 128] = 129
    d = (torch.randn(count, device="cuda", generator=gen).abs() * scale).to(torch.float16)
    b[:, at:at + 2] = d.view(torch.uint8).view(count, 2)
    return b


def _matrix(fmt, rows, cols, gen):
    return _blocks(fmt, rows * cols // FORMATS[fmt][1], gen).view(-1)


def _arena(case, gen):
    """experts + shared packed experts, gate | up | down each."""
    e = case["experts"] + SHARED
    size, up, down = _expert(case)
    a = torch.empty((e, size), dtype=torch.uint8, device="cuda")
    h, f = case["hidden"], case["ff"]
    a[:, :down] = _matrix(case["gate"], e * 2 * f, h, gen).view(e, -1)
    a[:, down:] = _matrix(case["down"], e * h, f, gen).view(e, -1)
    return a


def _zipf_logits(rng, tokens, experts):
    rank = rng.permutation(experts) + 1
    return (rng.standard_normal((tokens, experts)) - 1.1 * np.log(rank)[None, :]).astype(np.float32)


def _capture(fn):
    """A graph of fn's launches, after one eager pass that sizes the scratch."""
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        q4mi.use_torch_stream()
        fn()
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        q4mi.use_torch_stream()
        fn()
    q4mi.use_torch_stream()
    return g


def prepare(case, seed):
    lib = q4mi.lib()
    q4mi.use_torch_stream()
    lib.q4_hip_moe_scratch_warm()
    lib.q4_mmvq_warm()
    s = _PREPARE[case["kind"]](case, seed)
    s["case"] = case
    if case.get("graph", case["kind"] in ("decode", "window")):
        s["graph"] = _capture(lambda: _RUN[case["kind"]](s))
    return s


def run(state):
    if "graph" in state:
        state["graph"].replay()
        return state["out"]
    return _RUN[state["case"]["kind"]](state)


# -- gemv

def _prepare_gemv(case, seed):
    gen = _gen(seed)
    w = [_matrix(case["type"], case["rows"], case["cols"], gen) for _ in range(case["mats"])]
    x = torch.randn((case["mats"], case["n"], case["cols"]), device="cuda", generator=gen)
    y = torch.empty((case["mats"], case["n"], case["rows"]), device="cuda")
    return {"w": w, "x": x, "y": y, "out": {"y": y}}


def _run_gemv(s):
    c, lib = s["case"], q4mi.lib()
    ty = FORMATS[c["type"]][0]
    for i, w in enumerate(s["w"]):
        q4mi.check(lib.q4_mmvq_n(ty, w.data_ptr(), c["rows"], c["cols"], s["x"][i].data_ptr(),
                                 s["y"][i].data_ptr(), 1.0, c["n"]), "q4_mmvq_n")
    return s["out"]


# -- decode

def _prepare_decode(case, seed):
    gen, rng = _gen(seed), np.random.default_rng(seed)
    n, e, h, k = case["layers"], case["experts"], case["hidden"], case["topk"]
    s = {"arena": [_arena(case, gen) for _ in range(n)],
         "x": torch.randn((n, h), device="cuda", generator=gen),
         "y": torch.empty((n, h), device="cuda")}
    s["out"] = {"y": s["y"]}
    if case["routed"]:
        # router rows of about 1/sqrt(hidden), so logits are about N(0,1)
        s["router"] = torch.randn((n, e, h), device="cuda", generator=gen) / math.sqrt(h)
        s["gate"] = torch.randn((n, h), device="cuda", generator=gen) / math.sqrt(h)
        s["logits"] = torch.empty((n, e), device="cuda")
        s["sg"] = torch.empty((n, 1), device="cuda")
        s["ids"] = torch.empty((n, 64), dtype=torch.int32, device="cuda")
        s["wts"] = torch.empty((n, 64), device="cuda")
        s["count"] = torch.empty((n, 1), dtype=torch.int32, device="cuda")
        s["out"]["logits"] = s["logits"]
    else:
        s["lists"] = [_pick(rng.standard_normal((1, e)).astype(np.float32), k, e) for _ in range(n)]
    return s


def _pick(logits, k, shared):
    """ids and weights [tokens][k + 1]: softmax top-k, renormalised, and the
    shared expert at weight 1."""
    p = np.exp(logits.astype(np.float64) - logits.max(axis=1, keepdims=True))
    ids = np.argsort(-p, axis=1, kind="stable")[:, :k]
    w = np.take_along_axis(p, ids, axis=1)
    w /= w.sum(axis=1, keepdims=True)
    t = len(ids)
    return (np.ascontiguousarray(np.concatenate([ids, np.full((t, 1), shared)], 1), np.int32),
            np.ascontiguousarray(np.concatenate([w, np.ones((t, 1))], 1), np.float32))


def _run_decode(s):
    c, lib = s["case"], q4mi.lib()
    size, up, down = _expert(c)
    gt, dt = FORMATS[c["gate"]][0], FORMATS[c["down"]][0]
    e, h, f, k = c["experts"], c["hidden"], c["ff"], c["topk"]
    s["y"].zero_()
    for i in range(c["layers"]):
        base, x, y = s["arena"][i].data_ptr(), s["x"][i].data_ptr(), s["y"][i].data_ptr()
        if c["routed"]:
            ok = lib.q4mi_moe_route_exec(
                s["router"][i].data_ptr(), 0, s["gate"][i].data_ptr(), x, h, e, k,
                s["logits"][i].data_ptr(), s["ids"][i].data_ptr(), s["wts"][i].data_ptr(),
                s["count"][i].data_ptr(), e, s["sg"][i].data_ptr(), base, size, gt, 0, gt, up,
                dt, down, y, f)
        else:
            ids, wts = s["lists"][i]
            ok = lib.q4_hip_moe_exec(
                base, size, ids.ctypes.data_as(ctypes.c_void_p),
                wts.ctypes.data_as(ctypes.c_void_p), ids.shape[1], gt, 0, gt, up, dt, down, x,
                None, None, None, y, f, h, h)
        q4mi.check(ok, "decode layer")
    return s["out"]


# -- window

def _prepare_window(case, seed):
    gen, rng = _gen(seed), np.random.default_rng(seed)
    n, t, e, h, k = (case[q] for q in ("layers", "tokens", "experts", "hidden", "topk"))
    s = {"arena": [_arena(case, gen) for _ in range(n)],
         "x": torch.randn((n, t, h), device="cuda", generator=gen),
         "y": torch.empty((n, t, h), device="cuda"),
         "ids": torch.full((n, t, 64), -1, dtype=torch.int32, device="cuda"),
         "wts": torch.zeros((n, t, 64), device="cuda"),
         "count": torch.full((n, t), k + SHARED, dtype=torch.int32, device="cuda")}
    for i in range(n):
        ids, wts = _pick(rng.standard_normal((t, e)).astype(np.float32), k, e)
        s["ids"][i, :, :k + SHARED] = torch.from_numpy(ids).cuda()
        s["wts"][i, :, :k + SHARED] = torch.from_numpy(wts).cuda()
    s["out"] = {"y": s["y"]}
    return s


def _run_window(s):
    c, lib = s["case"], q4mi.lib()
    size, up, down = _expert(c)
    gt, dt = FORMATS[c["gate"]][0], FORMATS[c["down"]][0]
    s["y"].zero_()
    for i in range(c["layers"]):
        q4mi.check(lib.q4_hip_moe_exec_win(
            s["arena"][i].data_ptr(), size, s["ids"][i].data_ptr(), s["wts"][i].data_ptr(),
            s["count"][i].data_ptr(), c["tokens"], gt, 0, gt, up, dt, down, s["x"][i].data_ptr(),
            None, s["y"][i].data_ptr(), c["ff"], c["hidden"], c["hidden"]), "window layer")
    return s["out"]


# -- prefill

def _prepare_prefill(case, seed):
    gen, rng = _gen(seed), np.random.default_rng(seed)
    t, e, h, f, k = (case[q] for q in ("tokens", "experts", "hidden", "ff", "topk"))
    lib, rows, i32 = q4mi.lib(), t * k, torch.int32
    new = lambda *n, dtype=torch.float32: torch.empty(n, dtype=dtype, device="cuda")  # noqa: E731
    s = {"arena": _arena(case, gen), "x": torch.randn((t, h), device="cuda", generator=gen),
         "logits": torch.from_numpy(_zipf_logits(rng, t, e)).cuda(),
         "ids": new(t, k, dtype=i32), "wts": new(t, k), "a_tok": new(rows + t, dtype=i32),
         "rsrc": new(rows, dtype=i32), "rw": new(rows), "stg": new(512, dtype=i32),
         "stgn": new(1, dtype=i32), "ek": new(512, dtype=i32), "bounds": new(e + 2, dtype=i32),
         "xq": new(int(lib.q4_mmq_q8_bytes(t, h)), dtype=torch.uint8),
         "hq": new(int(lib.q4_mmq_q8_bytes(rows + t, f)), dtype=torch.uint8),
         "pd": new(rows + t, h), "y": new(t, h)}
    # the shared expert's rows (every token) follow the routed pack
    s["a_tok"][rows:] = torch.arange(t, dtype=i32, device="cuda")
    s["bounds"][e + 1] = rows + t
    s["out"] = {"y": s["y"], "ids": s["ids"], "wts": s["wts"]}
    return s


def _run_prefill(s):
    c, lib = s["case"], q4mi.lib()
    p = {n: v.data_ptr() for n, v in s.items() if isinstance(v, torch.Tensor)}
    t, e, h, f, k = (c[q] for q in ("tokens", "experts", "hidden", "ff", "topk"))
    size, _, down = _expert(c)
    gt, dt = FORMATS[c["gate"]][0], FORMATS[c["down"]][0]
    rows, shared = t * k, p["arena"] + e * size
    s["y"].zero_()
    q4mi.check(lib.q4_hip_route_pf(p["logits"], p["ids"], p["wts"], t, e, k), "route")
    q4mi.check(lib.q4mi_assign(p["ids"], p["wts"], p["a_tok"], p["rsrc"], p["rw"], p["stg"],
                               p["stgn"], p["ek"], p["bounds"], t, k, e, t), "pack")
    q4mi.check(lib.q4_mmq_quantize(p["x"], None, p["xq"], gt, h, t), "quantize")
    q4mi.check(lib.q4mi_mmq_gate_up_x(p["arena"], shared, gt, f, h, size, e, p["xq"], t,
                                      p["a_tok"], p["bounds"], rows + t, p["hq"]), "gate/up")
    q4mi.check(lib.q4mi_mmq_mul_id_x(p["arena"] + down, shared + down, dt, h, f, size, e, p["hq"],
                                     p["bounds"], rows + t, p["pd"], h), "down")
    q4mi.check(lib.q4mi_expert_reduce_x(p["y"], p["pd"], p["rsrc"], p["rw"], t, k, h, rows, None),
               "reduce")
    return s["out"]


# -- fp16-activation prefill

def _prepare_xg(case, seed):
    gen, rng = _gen(seed), np.random.default_rng(seed)
    t, e, h, f, k = (case[q] for q in ("tokens", "experts", "hidden", "ff", "topk"))
    lib, rows = q4mi.lib(), t * k
    ids, wts = _pick(_zipf_logits(rng, t, e), k, e)
    ids, wts = ids[:, :k], wts[:, :k]
    # the pack and its tile table, which the engine builds on the host
    order = np.argsort(ids.reshape(-1), kind="stable")
    rsrc = np.empty(rows, np.int32)
    rsrc[order] = np.arange(rows, dtype=np.int32)
    a_tok = np.concatenate([order // k, np.arange(t)]).astype(np.int32)
    ek = np.append(np.bincount(ids.reshape(-1), minlength=e), t).astype(np.uint32)
    first = np.concatenate([[0], np.cumsum(ek)[:-1]]).astype(np.uint32)
    slot = np.arange(e + 1, dtype=np.int32)
    cap = lib.q4_xg_tile_cap(rows + t, e + 1)
    tiles = np.zeros(4 * cap, np.int32)
    nt = lib.q4_xg_tiles(ek.ctypes.data, first.ctypes.data, slot.ctypes.data, e + 1,
                         tiles.ctypes.data, cap)
    up = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()  # noqa: E731
    s = {"arena": _arena(case, gen), "x": torch.randn((t, h), device="cuda", generator=gen),
         "tiles": up(tiles[:4 * nt]), "a_tok": up(a_tok), "rsrc": up(rsrc),
         "rw": up(wts.reshape(-1)), "nt": nt,
         "x16": torch.empty((t, h), dtype=torch.float16, device="cuda"),
         "h16": torch.empty((rows + t, f), dtype=torch.float16, device="cuda"),
         "pd": torch.empty((rows + t, h), device="cuda"), "y": torch.empty((t, h), device="cuda")}
    s["out"] = {"y": s["y"]}
    return s


def _run_xg(s):
    c, lib = s["case"], q4mi.lib()
    p = {n: v.data_ptr() for n, v in s.items() if isinstance(v, torch.Tensor)}
    t, h, f, k = c["tokens"], c["hidden"], c["ff"], c["topk"]
    size, up, down = _expert(c)
    gt, dt = FORMATS[c["gate"]][0], FORMATS[c["down"]][0]
    s["y"].zero_()
    q4mi.check(lib.q4_xg_cvt(p["x"], p["x16"], t * h), "convert")
    q4mi.check(lib.q4_xg_gu(gt, p["arena"], size, 0, up, h, f, p["tiles"], s["nt"], p["x16"],
                            p["a_tok"], p["h16"]), "gate/up")
    q4mi.check(lib.q4_xg_dn(dt, p["arena"], size, down, f, h, p["tiles"], s["nt"], p["h16"],
                            p["pd"]), "down")
    q4mi.check(lib.q4mi_expert_reduce_x(p["y"], p["pd"], p["rsrc"], p["rw"], t, k, h, t * k, None),
               "reduce")
    return s["out"]


_PREPARE = {"gemv": _prepare_gemv, "decode": _prepare_decode, "window": _prepare_window,
            "prefill": _prepare_prefill, "xg": _prepare_xg}
_RUN = {"gemv": _run_gemv, "decode": _run_decode, "window": _run_window, "prefill": _run_prefill,
        "xg": _run_xg}


# ------------------------------------------------------- results in 64 bits
# Weights are dequantized from the formats' definitions, activations and h
# take the q8 rounding that the path is defined by (32-value groups: d =
# amax/127 and 127/amax in fp32, round to nearest even), and every product
# and sum is in fp64.  The codebooks are the formats' tables, read as data.

def _codes(header, name):
    text = open(os.path.join("include", header)).read().replace("\\\n", " ")
    body = re.search(r"#define %s\s+([^\n]*)" % name, text).group(1)
    return torch.tensor([int(v, 16) for v in re.findall(r"0x[0-9a-fA-F]+", body)], device="cuda")


def _grid(fmt):
    if fmt == "IQ3_S":
        return 2 * ((_codes("q4mi_iq3s_grid.h", "Q4MI_IQ3S_CODES")[:, None]
                     >> (3 * torch.arange(4, device="cuda"))) & 7) + 1
    if fmt == "IQ2_S":
        level = torch.tensor([8, 25, 43, 0], device="cuda")
        return level[(_codes("q4mi_iq2s_grid.h", "Q4MI_IQ2S_CODES")[:, None]
                      >> (2 * torch.arange(8, device="cuda"))) & 3]
    level = torch.tensor([4, 12, 20, 28, 36, 44, 52, 62], device="cuda")   # IQ3_XXS
    return level[(_codes("q4mi_iqxx_grids.h", "Q4MI_IQ3XXS_CODES")[:, None]
                  >> (3 * torch.arange(4, device="cuda"))) & 7]


def _bits(b, n):
    """The low n bits of every element, one more axis."""
    return (b[..., None] >> torch.arange(n, device="cuda")) & 1


def _decode(fmt, raw):
    """raw [blocks][bytes] -> integers [blocks][values] without the sub-block
    multipliers, the multipliers [blocks][values], the block scales [blocks]."""
    _, vals, size, at, _ = FORMATS[fmt]
    b = raw.to(torch.int64)
    n = len(b)
    d = raw[:, at:at + 2].contiguous().view(torch.float16).view(n).double()
    one = torch.ones((n, 1), dtype=torch.int64, device="cuda")
    nl = torch.tensor([-127, -104, -83, -65, -49, -35, -22, -10, 1, 13, 25, 38, 53, 69, 89, 113],
                      device="cuda")
    nib = lambda v: torch.stack([v & 15, v >> 4], -1).reshape(n, -1)   # noqa: E731
    if fmt == "Q8_0":
        return (b[:, 2:] ^ 128) - 128, one, d
    if fmt == "IQ4_NL":
        return nl[torch.cat([b[:, 2:] & 15, b[:, 2:] >> 4], 1)], one, d
    if fmt == "Q2_0":
        return ((b[:, 2:, None] >> (2 * torch.arange(4, device="cuda"))) & 3).reshape(n, -1) - 1, one, d
    if fmt == "IQ4_XS":
        q = b[:, 8:].view(n, 8, 16)
        hi = (b[:, 2] | (b[:, 3] << 8))[:, None] >> (2 * torch.arange(8, device="cuda")) & 3
        m = (nib(b[:, 4:8]) | (hi << 4)) - 32
        return nl[torch.cat([q & 15, q >> 4], 2)].reshape(n, -1), m.repeat_interleave(32, 1), d
    if fmt == "Q6_K":
        ql, qh = b[:, :128].view(n, 2, 2, 32), b[:, 128:192].view(n, 2, 1, 32)
        lo = torch.cat([ql & 15, ql >> 4], 2)
        hi = (qh >> (2 * torch.arange(4, device="cuda")).view(1, 1, 4, 1)) & 3
        m = ((b[:, 192:208] ^ 128) - 128).repeat_interleave(16, 1)
        return ((lo | (hi << 4)) - 32).reshape(n, -1), m, d
    if fmt == "IQ3_S":
        idx = b[:, 2:66] | (_bits(b[:, 66:74], 8).reshape(n, 64) << 8)
        sign = 1 - 2 * _bits(b[:, 74:106], 8).reshape(n, 256)
        m = 2 * nib(b[:, 106:110]) + 1
        return _grid(fmt)[idx].reshape(n, 256) * sign, m.repeat_interleave(32, 1), d
    if fmt == "IQ2_S":
        hi = (b[:, 66:74, None] >> (2 * torch.arange(4, device="cuda"))) & 3
        idx = b[:, 2:34] | (hi.reshape(n, 32) << 8)
        sign = 1 - 2 * _bits(b[:, 34:66], 8).reshape(n, 256)
        m = 2 * nib(b[:, 74:82]) + 1
        return _grid(fmt)[idx].reshape(n, 256) * sign, m.repeat_interleave(16, 1), d * 0.125
    q = b[:, 66:98].view(n, 8, 4)                                          # IQ3_XXS
    aux = q[..., 0] | (q[..., 1] << 8) | (q[..., 2] << 16) | (q[..., 3] << 24)
    s7 = _bits((aux[..., None] >> (7 * torch.arange(4, device="cuda"))) & 127, 7)
    sign = 1 - 2 * torch.cat([s7, s7.sum(-1, keepdim=True) & 1], -1).reshape(n, 256)
    m = 2 * (aux >> 28) + 1
    return _grid(fmt)[b[:, 2:66]].reshape(n, 256) * sign, m.repeat_interleave(32, 1), d * 0.25


def _dequant(fmt, raw, cols):
    v, m, d = _decode(fmt, raw.view(-1, FORMATS[fmt][2]))
    return ((v * m).double() * d[:, None]).view(-1, cols)


def _f32(v):
    return v.float().double()


def _q8(x):
    """The q8 rounding of fp32 rows, as fp64 values."""
    g = _f32(x).view(-1, 32)
    a = g.abs().amax(1, keepdim=True)
    inv = torch.where(a > 0, _f32(127.0 / a.clamp(min=1e-45)), torch.zeros_like(a))
    q = _f32(g * inv).round().clamp(-128, 127)
    return (q * _f32(a / 127.0)).view(x.shape)


def _parts(case, packed):
    """gate, up and down of one packed expert in fp64."""
    _, up, down = _expert(case)
    return (_dequant(case["gate"], packed[:up], case["hidden"]),
            _dequant(case["gate"], packed[up:down], case["hidden"]),
            _dequant(case["down"], packed[down:], case["ff"]))


def _layer(case, arena, x, ids, wts):
    """sum_k wts[t][k] FFN_ids[t][k](x[t]) of one layer, fp64."""
    xq, y = _q8(x), torch.zeros(x.shape, dtype=torch.float64, device="cuda")
    for e in torch.unique(ids).tolist():
        t, k = torch.nonzero(ids == e, as_tuple=True)
        gate, up, down = _parts(case, arena[e])
        g, u = xq[t] @ gate.T, xq[t] @ up.T
        out = _q8(g / (1 + torch.exp(-g)) * u) @ down.T
        y.index_add_(0, t, out * wts[t, k].double()[:, None])
    return y


def _top(logits, k):
    p = torch.softmax(logits.double(), 1)
    w, ids = torch.sort(p, dim=1, descending=True, stable=True)
    return ids[:, :k], w[:, :k] / w[:, :k].sum(1, keepdim=True)


def _with_shared(case, ids, wts, weight):
    t = len(ids)
    return (torch.cat([ids, torch.full((t, 1), case["experts"], device="cuda")], 1),
            torch.cat([wts, weight.expand(t, 1)], 1))


def _fp16_weights(fmt, raw, cols):
    """The fp16 operands of the fp16-activation path: 256 times the weight,
    the scaled multiplier and the product each rounded to fp16."""
    v, m, d = _decode(fmt, raw.view(-1, FORMATS[fmt][2]))
    scale = (d[:, None] * m * 256.0).to(torch.float16).double()
    return ((v.double() * scale).to(torch.float16).double() / 256.0).view(-1, cols)


def exact(case, seed):
    s = _PREPARE[case["kind"]](case, seed)
    kind = case["kind"]
    if kind == "gemv":
        y = torch.empty(s["y"].shape, dtype=torch.float64, device="cuda")
        step = max(1, (1 << 25) // case["cols"])
        rb = _row_bytes(case["type"], case["cols"])
        for i, w in enumerate(s["w"]):
            xq = _q8(s["x"][i])
            for r in range(0, case["rows"], step):
                raw = w[r * rb:(r + step) * rb]
                y[i][:, r:r + step] = xq @ _dequant(case["type"], raw, case["cols"]).T
        return {"y": y}
    if kind == "decode":
        y, logits = [], []
        for i in range(case["layers"]):
            x = s["x"][i][None]
            if case["routed"]:
                lg = x.double() @ s["router"][i].double().T
                logits.append(lg[0])
                sg = torch.sigmoid(x.double() @ s["gate"][i].double())[:, None]
                ids, wts = _with_shared(case, *_top(lg, case["topk"]), sg)
            else:
                ids, wts = (torch.from_numpy(v).cuda() for v in s["lists"][i])
            y.append(_layer(case, s["arena"][i], x, ids, wts)[0])
        out = {"y": torch.stack(y)}
        if case["routed"]:
            out["logits"] = torch.stack(logits)
        return out
    if kind == "window":
        k = case["topk"] + SHARED
        return {"y": torch.stack([_layer(case, s["arena"][i], s["x"][i], s["ids"][i][:, :k],
                                         s["wts"][i][:, :k]) for i in range(case["layers"])])}
    if kind == "prefill":
        ids, wts = _top(s["logits"], case["topk"])
        one = torch.ones((1, 1), dtype=torch.float64, device="cuda")
        y = _layer(case, s["arena"], s["x"], *_with_shared(case, ids, wts, one))
        return {"y": y, "ids": ids.to(torch.int32), "wts": wts}
    # xg: rows of expert e are first[e] .. of the pack
    x16 = s["x"].to(torch.float16).double()
    y = torch.zeros(x16.shape, dtype=torch.float64, device="cuda")
    t, k, e = case["tokens"], case["topk"], case["experts"]
    tok, w = s["a_tok"].long(), torch.ones(t * k + t, dtype=torch.float64, device="cuda")
    w[s["rsrc"].long()] = s["rw"].double()
    _, up, down = _expert(case)
    tiles = s["tiles"].view(-1, 4)
    for expert in torch.unique(tiles[:, 3]).tolist():
        mine = tiles[tiles[:, 3] == expert]
        first, n = int(mine[0, 0]), int(mine[:, 1].sum())
        rows, raw = torch.arange(first, first + n, device="cuda"), s["arena"][expert]
        g, u = (x16[tok[rows]] @ _fp16_weights(case["gate"], part, case["hidden"]).T
                for part in (raw[:up], raw[up:down]))
        h = (g / (1 + torch.exp(-g)) * u).float().to(torch.float16).double()
        out = h @ _fp16_weights(case["down"], raw[down:], case["ff"]).T
        y.index_add_(0, tok[rows], out * w[rows][:, None])
    return {"y": y}
