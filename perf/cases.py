"""What a program that uses libdramamoe.so has it do, as cases that can be timed and compared.

Every case goes through the entry points of include/drama_moe.h as dramamoe.py binds them, on
layers of the one shape the library serves (hidden 2048, intermediate 512, 256 experts, top-8) with
the values of the benchmark configurations, in both scale encodings: "ref" (f16 pairs, int8 groups
of 128: a converted checkpoint) and "cfg" (bf16 pairs, one int8 scale per row).

Paths:
  step     dr_moe_decode_step*: one token through `layers` layers in one launch
  chain    the reference engine's launches of a decode step, per layer: dr_router_topk, dr_moe_decode*
  rows     a few tokens decoded together: router and experts of `rows` independent rows
  prefill  one layer of a prompt chunk as MoeStack.prefill issues it (router GEMM, top-k with the
           grouping, grouped experts, combine, shared expert on a second stream)
  engine   the same layer through the calls the reference engine itself makes (src/engine.rs:544-604),
           its host-side scan of the counts included
  dense    the int8 projections and the lm_head around the MoE
"""
import ctypes
import math
import os
import sys

import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "drama-rs_amd"))
import dramamoe as D  # noqa: E402

H, I, E, TOPK, EPS = 2048, 512, 256, 8, 1e-6
P = D.ptr
LAYER_KEYS = ("router", "nw", "gu_q", "gu_s", "d_q", "d_s", "sgu_q", "sgu_s", "sd_q", "sd_s")  # dr_decode_layer order


# ---- cases ------------------------------------------------------------------------------------


def listed():
    return [
        # the smallest call: an engine that runs attention between the MoE layers launches each alone
        {"name": "step_q4_1", "path": "step", "kind": "q4", "fmt": "ref", "layers": 1},
        # one token through the whole 40-layer model
        {"name": "step_q4_40", "path": "step", "kind": "q4", "fmt": "cfg", "layers": 40},
        # the block-FP8 experts of the original checkpoint, the part of the model kept in HBM
        {"name": "step_fp8_10", "path": "step", "kind": "fp8", "fmt": "ref", "layers": 10},
        # the reference engine relinked: its own launch sequence, per layer
        {"name": "chain_q4_8", "path": "chain", "kind": "q4", "fmt": "ref", "layers": 8},
        # a batch of speech streams decoded together, and a small one
        {"name": "rows_q4_20", "path": "rows", "kind": "q4", "fmt": "ref", "rows": 20},
        {"name": "rows_fp8_4", "path": "rows", "kind": "fp8", "fmt": "cfg", "rows": 4},
        # a short text prompt
        {"name": "prefill_q4_37", "path": "prefill", "kind": "q4", "fmt": "ref", "rows": 37, "packed": False, "skew": False},
        # the usual prompt with a reference voice
        {"name": "prefill_q4_300", "path": "prefill", "kind": "q4", "fmt": "cfg", "rows": 300, "packed": True, "skew": False},
        # the reference engine's prompt chunk through its own calls
        {"name": "engine_q4_512", "path": "engine", "kind": "q4", "fmt": "ref", "rows": 512},
        # the longest chunk (8192 pairs), on the tile-step copy
        {"name": "prefill_q4_1024", "path": "prefill", "kind": "q4", "fmt": "ref", "rows": 1024, "packed": True, "skew": False},
        # a routing with hot experts
        {"name": "prefill_fp8_600_skew", "path": "prefill", "kind": "fp8", "fmt": "ref", "rows": 600, "packed": True, "skew": True},
        # an int8 projection and the lm_head of one token
        {"name": "dense_lm_head", "path": "dense", "fmt": "cfg", "n": 151936},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    path = rng.choice(["step", "chain", "rows", "prefill", "prefill", "prefill", "engine", "dense"])
    kind, fmt = rng.choice(["q4", "q4", "fp8"]), rng.choice(["ref", "cfg"])
    if path == "step":
        return {"path": path, "kind": kind, "fmt": fmt, "layers": _log(rng, 1, 40 if kind == "q4" else 20)}
    if path == "chain":
        return {"path": path, "kind": kind, "fmt": fmt, "layers": _log(rng, 1, 12)}
    if path == "rows":
        return {"path": path, "kind": kind, "fmt": fmt, "rows": _log(rng, 1, 64)}
    if path == "prefill":
        return {"path": path, "kind": kind, "fmt": fmt, "rows": _log(rng, 2, 1024 if kind == "q4" else 600),
                "packed": rng.random() < 0.5, "skew": rng.random() < 0.3}
    if path == "engine":
        return {"path": path, "kind": kind, "fmt": "ref", "rows": _log(rng, 8, 512)}
    return {"path": path, "fmt": fmt, "n": _log(rng, 1000, 151936)}


# ---- weights ----------------------------------------------------------------------------------


def _bytes(n, gen):
    """n random bytes, n % 8 == 0."""
    return torch.randint(-(1 << 62), (1 << 62) - 1, (n // 8,), generator=gen, device="cuda").mul_(3).view(torch.uint8)


def _randn(shape, gen, dtype=torch.float32):
    return torch.randn(shape, generator=gen, device="cuda", dtype=dtype)


def _experts(n, k, case, gen):
    """(weights, scales) of the E routed experts, each [n, k]."""
    ref = case["fmt"] == "ref"
    if case["kind"] == "q4":  # nibbles uniform 0..15, scale |N(0, 0.02)| + 1e-4, min N(0, 0.02) per 64 inputs
        q = _bytes(E * n * k // 2, gen).view(E, n, k // 2)
        sm = _randn((E, n, k // 64, 2), gen, torch.float16 if ref else torch.bfloat16).mul_(0.02)
        sm[..., 0].abs_().add_(1e-4)
        return q, sm
    # e4m3 codes of values N(0, 100), block scales around 0.02 / 100
    q = torch.empty(E, n, k, dtype=torch.uint8, device="cuda")
    for e in range(0, E, 32):
        q[e:e + 32] = _randn((32, n, k), gen, torch.float16).mul_(100).clamp_(-448, 448).to(torch.float8_e4m3fn).view(torch.uint8)
    s = _randn((E, n // 128, k // 128), gen).abs_().mul_(0.02).add_(1e-4).div_(100)
    return q, s if ref else s.to(torch.bfloat16)


def _int8(n, k, fmt, gen):
    q = _bytes(n * k, gen).view(torch.int8).view(n, k).clamp_(min=-127)
    if fmt == "ref":
        return q, (_randn((n, k // 128), gen).abs_().mul_(0.02).add_(1e-4) / 73).half()
    return q, (_randn((n,), gen).abs_().mul_(0.02).add_(1e-4) / 73).to(torch.bfloat16)


def _layer(case, gen):
    L = {"router": (_randn((E + 1, H), gen) * 0.02).to(torch.bfloat16), "nw": 1 + 0.1 * _randn((H,), gen)}
    L["gu_q"], L["gu_s"] = _experts(2 * I, H, case, gen)
    L["d_q"], L["d_s"] = _experts(H, I, case, gen)
    L["sgu_q"], L["sgu_s"] = _int8(2 * I, H, case["fmt"], gen)
    L["sd_q"], L["sd_s"] = _int8(H, I, case["fmt"], gen)
    return L


def _pack(L, case, st):
    """L with its routed experts in the tile-step layout that prefill streams best."""
    lib, pk = D.lib(), dict(L)
    for q, s, n, k in (("gu_q", "gu_s", 2 * I, H), ("d_q", "d_s", H, I)):
        pk[q] = torch.empty_like(L[q])
        if case["kind"] == "q4":
            pk[s] = torch.empty_like(L[s])
            lib.dr_moe_pack_q4(P(L[q]), P(L[s]), E, n, k, P(pk[q]), P(pk[s]), st)
        else:
            lib.dr_moe_pack_fp8(P(L[q]), E, n, k, P(pk[q]), st)
    return pk


# ---- state ------------------------------------------------------------------------------------

_streams = []
_handles = {}


def _stream(i):
    """The program's streams: 0 carries every call in order, 1 the shared expert beside it."""
    while len(_streams) < 2:
        _streams.append(torch.cuda.Stream())
    return _streams[i]


def _gemm_handle(sp):
    """The GEMM handle of stream sp, kept for the process's lifetime as the engine keeps its own."""
    if sp not in _handles:
        h = ctypes.c_void_p()
        D.lib().dr_cublas_create(ctypes.byref(h), sp)
        _handles[sp] = h.value
    return _handles[sp]


class _State:
    pass


def _z(*shape, dtype=torch.float32):
    return torch.zeros(shape, dtype=dtype, device="cuda")


def _inputs(case, gen):
    """The activations of a case."""
    rows = case.get("rows", 1)
    x = _randn((rows, H), gen)
    out = {"x": x}
    if case["path"] in ("prefill", "engine"):
        out["hn"] = _randn((rows, H), gen).to(torch.bfloat16)
    if case.get("skew"):  # a tenth of the experts get half of the pairs, the picks of a row distinct
        hot = torch.randperm(E, generator=gen, device="cuda")[: E // 10]
        w = torch.ones(E, device="cuda")
        w[hot] = (E - hot.numel()) / hot.numel()
        out["idx"] = torch.multinomial(w.expand(rows, E), TOPK, generator=gen).to(torch.int32)
        wt = torch.rand(rows, TOPK, generator=gen, device="cuda") + 0.1
        out["wts"] = wt / wt.sum(1, keepdim=True)
        out["sg"] = _randn((rows,), gen)
    return out


def _layers(case):
    return case.get("layers", 1)


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed * 7919 + 1)
    s = _State()
    s.case = case
    sp = _stream(0).cuda_stream
    if case["path"] == "dense":
        s.x = _randn((H,), gen)
        s.nw = 1 + 0.1 * _randn((H,), gen)
        s.pq, s.ps = _int8(H, H, case["fmt"], gen)
        s.hq, s.hs = _int8(case["n"], H, case["fmt"], gen)
        s.h, s.y = _z(H), _z(case["n"])
        torch.cuda.synchronize()
        return s
    s.layers = [_layer(case, gen) for _ in range(_layers(case))]
    for k, v in _inputs(case, gen).items():
        setattr(s, k, v)
    rows = case.get("rows", 1)
    n = rows * TOPK
    torch.cuda.synchronize()
    if case["path"] == "step":
        s.table = torch.tensor([[L[k].data_ptr() for k in LAYER_KEYS] for L in s.layers], dtype=torch.int64, device="cuda")
        s.ll, s.sync = _z(D.STEP_LL_WORDS, dtype=torch.int64), _z(4, dtype=torch.int32)
        s.idx, s.wts = _z(len(s.layers), TOPK, dtype=torch.int32), _z(len(s.layers), TOPK)
        s.sg, s.xs = _z(len(s.layers)), _z(len(s.layers), H)
    else:
        s.logits, s.counter = _z(rows, E + 1), _z(4, dtype=torch.int32)
        if not case.get("skew"):
            s.idx, s.wts, s.sg = _z(rows, TOPK, dtype=torch.int32), _z(rows, TOPK), _z(rows)
    if case["path"] in ("chain", "rows"):
        s.act, s.y, s.tags = _z(rows, TOPK + 1, I), _z(rows, H), _z(896, dtype=torch.int64)
    if case["path"] in ("prefill", "engine"):
        s.counts, s.offsets = _z(E, dtype=torch.int32), _z(E, dtype=torch.int32)
        s.slot_of, s.row_of_slot = _z(n, dtype=torch.int32), _z(n + 16, dtype=torch.int32)
        s.act, s.yp = _z(n, I, dtype=torch.bfloat16), _z(n, H)
        s.sact, s.sh = _z(rows, I, dtype=torch.bfloat16), _z(rows, H)
        s.gemm = _gemm_handle(sp)
    if case["path"] == "prefill":
        s.W = _pack(s.layers[0], case, sp) if case["packed"] else s.layers[0]
        s.fork, s.join = torch.cuda.Event(), torch.cuda.Event()
        if case["packed"]:
            torch.cuda.synchronize()
            for k in ("gu_q", "d_q"):  # this program decodes elsewhere: only the copy is kept
                s.layers[0][k] = None
    if case["path"] == "engine":
        s.fill, s.xp = _z(E, dtype=torch.int32), _z(n, H, dtype=torch.bfloat16)
        s.wbuf, s.hh = _z(2 * I, H, dtype=torch.bfloat16), _z(rows, 2 * I)
        s.host = torch.zeros(2, E, dtype=torch.int32, pin_memory=True)
    torch.cuda.synchronize()
    return s


# ---- one pass ---------------------------------------------------------------------------------


def _sfx(case):
    return ("_fp8" if case["kind"] == "fp8" else "") + ("" if case["fmt"] == "ref" else "_bf16s")


def _experts_args(L):
    return tuple(P(L[k]) for k in ("gu_q", "gu_s", "d_q", "d_s"))


def _shared_args(L):
    return tuple(P(L[k]) for k in ("sgu_q", "sgu_s", "sd_q", "sd_s"))


def _run_step(s, lib, sp):
    f = getattr(lib, "dr_moe_decode_step" + _sfx(s.case))
    f(P(s.table), len(s.layers), P(s.x), E, H, I, TOPK, EPS, P(s.ll), P(s.sync), P(s.idx), P(s.wts), P(s.sg), P(s.xs),
      None, 0, sp)
    return {"x": s.x, "idx": s.idx, "wts": s.wts, "sgate": s.sg, "xs": s.xs}


def _run_chain(s, lib, sp):
    yb = () if s.case["fmt"] == "ref" else (None,)
    f = getattr(lib, "dr_moe_decode" + _sfx(s.case))
    for L in s.layers:
        lib.dr_router_topk(P(L["router"]), P(s.x), P(L["nw"]), EPS, P(s.logits), E, TOPK, H, P(s.idx), P(s.wts), P(s.sg),
                           P(s.counter), None, None, None, None, 0, 0, 0, 0, sp)
        f(*_experts_args(L), *_shared_args(L), P(s.x), P(s.idx), P(s.wts), P(s.sg), P(s.x), P(s.act), P(s.x), *yb, H, I,
          TOPK, P(L["nw"]), EPS, None, 0, sp)
    return {"x": s.x, "idx": s.idx, "wts": s.wts, "logits": s.logits}


def _run_rows(s, lib, sp):
    rows, L = s.case["rows"], s.layers[0]
    yb = () if s.case["fmt"] == "ref" else (None,)
    if s.case["kind"] == "fp8":
        f = getattr(lib, "dr_moe_decode_rows_routed" + _sfx(s.case))
        f(P(L["router"]), P(L["nw"]), EPS, E, *_experts_args(L), *_shared_args(L), P(s.x), P(s.logits), P(s.idx),
          P(s.wts), P(s.sg), P(s.counter), P(s.tags), P(s.x), P(s.act), P(s.y), *yb, rows, H, I, TOPK, sp)
    else:
        for r in range(0, rows, 8):  # the router takes up to 8 rows a call
            lib.dr_router_topk_rows(P(L["router"]), P(s.x[r:]), P(L["nw"]), EPS, P(s.logits[r:]), E, TOPK, H,
                                    min(8, rows - r), P(s.idx[r:]), P(s.wts[r:]), P(s.sg[r:]), P(s.counter), sp)
        f = getattr(lib, "dr_moe_decode_rows" + _sfx(s.case))
        f(*_experts_args(L), *_shared_args(L), P(s.x), P(s.idx), P(s.wts), P(s.sg), P(s.x), P(s.act), P(s.y), *yb, rows,
          H, I, TOPK, P(L["nw"]), EPS, sp)
    return {"y": s.y, "idx": s.idx, "wts": s.wts, "logits": s.logits}


def _run_prefill(s, lib, sp):
    case, L, W = s.case, s.layers[0], s.W
    rows = case["rows"]
    main, side = _stream(0), _stream(1)
    overlap = rows >= 64  # for a few rows the events cost more than they save
    if overlap:
        s.fork.record(main)
        side.wait_event(s.fork)
    shared = lib.dr_moe_shared_prefill if case["fmt"] == "ref" else lib.dr_moe_shared_prefill_bf16s
    shared(*_shared_args(L), P(s.hn), rows, P(s.sact), P(s.sh), H, I, side.cuda_stream if overlap else sp)
    if overlap:
        s.join.record(side)
    if case["skew"]:
        lib.dr_moe_group_rows(P(s.idx), rows, TOPK, E, P(s.counts), P(s.offsets), P(s.slot_of), P(s.row_of_slot), sp)
    else:
        lib.dr_gemm(s.gemm, P(s.hn), P(L["router"]), P(s.logits), rows, E + 1, H, 0.0)
        lib.dr_moe_topk_group(P(s.logits), rows, E, TOPK, E + 1, P(s.idx), P(s.wts), P(s.sg), P(s.counts),
                              P(s.offsets), P(s.slot_of), P(s.row_of_slot), P(s.counter), sp)
    f = getattr(lib, "dr_moe_prefill_rows" + ("_packed" if case["packed"] else "") + _sfx(case))
    f(*_experts_args(W), P(s.hn), rows, P(s.row_of_slot), P(s.offsets), P(s.counts), P(s.act), P(s.yp), E, H, I, sp)
    if overlap:
        main.wait_event(s.join)
    lib.dr_moe_combine(P(s.x), P(s.yp), P(s.slot_of), P(s.wts), P(s.sg), P(s.sh), rows, TOPK, H, sp)
    return {"x": s.x, "idx": s.idx, "wts": s.wts, "sgate": s.sg, "shared": s.sh}


def _run_engine(s, lib, sp):
    case, L = s.case, s.layers[0]
    rows, n = case["rows"], case["rows"] * TOPK
    lib.dr_gemm(s.gemm, P(s.hn), P(L["router"]), P(s.logits), rows, E + 1, H, 0.0)
    lib.dr_moe_topk(P(s.logits), rows, E, TOPK, E + 1, P(s.idx), P(s.wts), P(s.sg), sp)
    lib.dr_dequant_q8(P(L["sgu_q"]), P(L["sgu_s"]), P(s.wbuf), 2 * I, H, sp)
    lib.dr_gemm(s.gemm, P(s.hn), P(s.wbuf), P(s.hh), rows, 2 * I, H, 0.0)
    lib.dr_swiglu_rows(P(s.hh), P(s.sact), rows, I, sp)
    lib.dr_dequant_q8(P(L["sd_q"]), P(L["sd_s"]), P(s.wbuf), H, I, sp)
    lib.dr_gemm(s.gemm, P(s.sact), P(s.wbuf), P(s.sh), rows, H, I, 0.0)
    lib.dr_memset(P(s.counts), 0, E * 4, sp)
    lib.dr_moe_count(P(s.idx), n, P(s.counts), sp)
    lib.dr_d2h(P(s.host), P(s.counts), E * 4, sp)
    lib.dr_stream_sync(sp)
    s.host[1].copy_(torch.cumsum(s.host[0], 0, dtype=torch.int32) - s.host[0])
    lib.dr_h2d(P(s.offsets), P(s.host[1]), E * 4, sp)
    lib.dr_memset(P(s.fill), 0, E * 4, sp)
    lib.dr_moe_permute(P(s.idx), rows, TOPK, P(s.offsets), P(s.fill), P(s.slot_of), P(s.hn), P(s.xp), H, sp)
    f = lib.dr_moe_prefill_fp8 if case["kind"] == "fp8" else lib.dr_moe_prefill
    f(*_experts_args(L), P(s.xp), P(s.offsets), P(s.counts), P(s.act), P(s.yp), E, H, I, sp)
    lib.dr_moe_combine(P(s.x), P(s.yp), P(s.slot_of), P(s.wts), P(s.sg), P(s.sh), rows, TOPK, H, sp)
    return {"x": s.x, "idx": s.idx, "wts": s.wts, "sgate": s.sg, "shared": s.sh, "logits": s.logits}


def _run_dense(s, lib, sp):
    n = s.case["n"]
    if s.case["fmt"] == "cfg":
        lib.dr_gemv_q8_bf16s(P(s.pq), P(s.ps), P(s.x), P(s.x), P(s.h), H, H, P(s.nw), EPS, sp)
        lib.dr_gemv_q8_bf16s(P(s.hq), P(s.hs), P(s.h), None, P(s.y), n, H, P(s.nw), EPS, sp)
    else:
        lib.dr_gemv_q8(P(s.pq), P(s.ps), P(s.x), P(s.x), P(s.h), H, H, P(s.nw), EPS, None, 0, sp)
        lib.dr_gemv_q8(P(s.hq), P(s.hs), P(s.h), None, P(s.y), n, H, P(s.nw), EPS, None, 0, sp)
    return {"h": s.h, "y": s.y}


_RUN = {"step": _run_step, "chain": _run_chain, "rows": _run_rows, "prefill": _run_prefill, "engine": _run_engine,
        "dense": _run_dense}


def run(s):
    return _RUN[s.case["path"]](s, D.lib(), _stream(0).cuda_stream)


# ---- what a pass cannot do without --------------------------------------------------------------


def work(case):
    ref = case["fmt"] == "ref"

    def int8(n, k):
        return n * k + (n * (k // 128) * 2 if ref else n * 2)

    if case["path"] == "dense":
        return {"bytes": int8(H, H) + int8(case["n"], H) + 4 * (3 * H + case["n"]), "flops": 2 * H * (H + case["n"])}
    if case["kind"] == "q4":
        expert = 3 * H * I // 2 + 3 * H * I // 64 * 4
    else:
        expert = 3 * H * I + 3 * H * I // 16384 * (4 if ref else 2)
    rows, layers = case.get("rows", 1), _layers(case)
    if case.get("skew"):
        hot = E // 10
        p = [0.5 * TOPK / hot, 0.5 * TOPK / (E - hot)]
        hit = hot * (1 - (1 - p[0]) ** rows) + (E - hot) * (1 - (1 - p[1]) ** rows)
    else:
        hit = E * (1 - (1 - TOPK / E) ** rows)
    weights = hit * expert + int8(2 * I, H) + int8(H, I) + (0 if case.get("skew") else (E + 1) * H * 2) + H * 4
    acts = rows * H * (2 * 4 + (2 if case["path"] in ("prefill", "engine") else 0))
    flops = 2 * rows * (3 * H * I * (TOPK + 1) + (0 if case.get("skew") else (E + 1) * H))
    return {"bytes": layers * (weights + acts), "flops": layers * flops}


def tolerance(case):
    # measured against exact(): decode 8e-7 at most, prefill 4e-5 (an activation whose bf16 rounding falls
    # the other way); four times that
    return {"rel": 2e-4 if case["path"] in ("prefill", "engine") else 4e-6}


# ---- the same in 64 bits ------------------------------------------------------------------------


def _deq_expert(q, s, kind):
    """One expert [n, k] in float64."""
    if kind == "q4":
        v = torch.stack([q & 15, q >> 4], -1).flatten(-2).double()  # low nibble first
        sm = s.double().repeat_interleave(64, 1)
        return v * sm[..., 0] + sm[..., 1]
    w = q.view(torch.float8_e4m3fn).float().double()
    return w * s.double().repeat_interleave(128, 0).repeat_interleave(128, 1)


def _deq_int8(q, s):
    s = s.double()
    return q.double() * (s.repeat_interleave(128, 1) if s.dim() == 2 else s[:, None])


def _norm(x, nw):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * nw.double()


def _bf16(t):
    return t.to(torch.bfloat16).double()


def _route(logits):
    p = torch.softmax(logits[:, :E], 1)
    w, idx = torch.topk(p, TOPK, dim=1)
    return idx, w / w.sum(1, keepdim=True), logits[:, E]


def _moe(L, kind, xn, idx, rnd):
    """[rows, TOPK, H]: every pick's expert output; rnd rounds the activations as the entry point states."""
    out = torch.zeros(xn.shape[0], TOPK, H, dtype=torch.float64, device="cuda")
    for e in torch.unique(idx).tolist():
        r, k = torch.nonzero(idx == e, as_tuple=True)
        gu = xn[r] @ _deq_expert(L["gu_q"][e], L["gu_s"][e], kind).T
        a = rnd(torch.nn.functional.silu(gu[:, :I]) * gu[:, I:])
        out[r, k] = a @ _deq_expert(L["d_q"][e], L["d_s"][e], kind).T
    return out


def _shared(L, xn, rnd, wrnd=lambda w: w):
    gu = xn @ wrnd(_deq_int8(L["sgu_q"], L["sgu_s"])).T
    return rnd(torch.nn.functional.silu(gu[:, :I]) * gu[:, I:]) @ wrnd(_deq_int8(L["sd_q"], L["sd_s"])).T


def exact(case, seed):
    if case["path"] == "dense":
        s = prepare(case, seed)
        x = s.x.double()
        h = x + _deq_int8(s.pq, s.ps) @ _norm(x, s.nw)
        hn = _norm(h, s.nw)
        y = torch.cat([_deq_int8(s.hq[i:i + 8192], s.hs[i:i + 8192]) @ hn for i in range(0, case["n"], 8192)])
        return {"h": h, "y": y}
    s = prepare(dict(case, packed=False) if case["path"] == "prefill" else case, seed)
    kind, keep = case["kind"], lambda t: t
    x = s.x.double()
    if case["path"] in ("prefill", "engine"):
        L, hn = s.layers[0], s.hn.double()
        logits = hn @ L["router"].double().T
        if case.get("skew"):
            idx, wts, sg = s.idx.long(), s.wts.double(), s.sg.double()
        else:
            idx, wts, sg = _route(logits)
        y = (wts[..., None] * _moe(L, kind, hn, idx, _bf16)).sum(1)
        sh = _shared(L, hn, _bf16, _bf16 if case["path"] == "engine" else keep)
        out = {"x": x + torch.sigmoid(sg)[:, None] * sh + y, "idx": None, "wts": wts, "sgate": sg, "shared": sh}
        if case["path"] == "engine":
            out["logits"] = logits
        return out
    wts_all, sg_all, xs = [], [], []
    for L in s.layers:
        xn = _norm(x, L["nw"])
        logits = xn @ L["router"].double().T
        idx, wts, sg = _route(logits)
        y = (wts[..., None] * _moe(L, kind, xn, idx, keep)).sum(1)
        x = x + torch.sigmoid(sg)[:, None] * _shared(L, xn, keep) + y
        wts_all.append(wts[0]), sg_all.append(sg[0]), xs.append(x[0])
    if case["path"] == "step":
        return {"x": x, "idx": None, "wts": torch.stack(wts_all), "sgate": torch.stack(sg_all), "xs": torch.stack(xs)}
    if case["path"] == "chain":
        return {"x": x, "idx": None, "wts": wts, "logits": logits}
    return {"y": x, "idx": None, "wts": wts, "logits": logits}
