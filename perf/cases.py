"""The work that a user of this package has it do, as cases that can be timed and compared.

Four kinds of call, each through the package's public entry points:
  layer      one fused MoE layer on packed weights (Context.layer), the path that inference runs: from fp16
             activations to fp16 outputs, or from the fp32 activations of the residual path (slot-scaled) into the
             hyper-connection streams
  recording  the same layer as the stage-by-stage recording on HF-layout weights (QwenMoe.moe_rec), for callers that
             keep their dispatch sequence
  stages     the routing and data-movement entry points by themselves (route, scan, scatter, combine)
  pack       one layer's checkpoint weights (bf16) into the packed layout (Context.pack_weights), paid once per layer
             that is loaded, and once per layer and pass where a model is streamed through the card

A case's fields: rows (tokens of the call), d, experts, topk, inter, shared (0, or the shared expert's width), act
("f16" or "f32" activations), hc (hyper-connection streams that the output goes into, 0: a plain fp16 output) and skew
(a Zipf-like router bias).
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.abspath("r-mda_amd"))
from rmda_moe import api  # noqa: E402

W_STD = 0.02            # expert and router weights
INJ_STRIDE, INJ_OFF = 384, 320  # the injection logits' row stride and first column
TILE = 128              # row tile of the drop-in stages

MID = dict(d=2048, experts=128, topk=8, inter=768, shared=0)
TEACHER = dict(d=2560, experts=512, topk=10, inter=640, shared=640)


def _case(kind, rows, shape, act="f16", hc=0, skew=False, **more):
    return dict(kind=kind, rows=rows, **shape, act=act, hc=hc, skew=skew, **more)


def listed():
    return [
        # one token of one sequence: the smallest call, its expert weights read for a single row
        _case("layer", 1, MID, name="token_1"),
        # a whole small layer: 256 tokens through 8 wide experts, bound by launches as much as by work
        _case("layer", 256, dict(d=512, experts=8, topk=2, inter=1024, shared=0), name="tiny_256"),
        # one sequence's 16-token block on the teacher's shape, as its forward pass calls it
        _case("layer", 16, TEACHER, act="f32", hc=4, name="teacher_block_16"),
        # eight sequences' 16-token blocks: weight streaming
        _case("layer", 128, MID, name="decode_128"),
        # the ragged last chunk of a prompt
        _case("layer", 777, MID, name="chunk_777"),
        # a training batch or a prompt of 8 x 256 tokens
        _case("layer", 2048, MID, name="prefill_2048"),
        # the same with a few experts taking most rows and many taking none
        _case("layer", 2048, MID, skew=True, name="skewed_2048"),
        # many small experts and a shared one, 16 x 256 tokens
        _case("layer", 4096, dict(d=2048, experts=512, topk=10, inter=512, shared=512), name="fine_shared_4096"),
        # the teacher's layer on a training batch, fp32 activations into its four streams
        _case("layer", 2048, TEACHER, act="f32", hc=4, name="teacher_2048"),
        # the same kind of batch through the stage-by-stage recording
        _case("recording", 2048, MID, act="f32", hc=4, name="recording_2048"),
        # the routing and data-movement stages as a caller's own sequence dispatches them
        _case("stages", 2048, MID, hc=4, name="stages_2048"),
        # the teacher's layer, from the checkpoint's bf16 to what the fused layer reads
        _case("pack", 2048, TEACHER, name="pack_teacher"),
    ]


def draw(rng):
    while True:
        kind = rng.choice(["layer"] * 6 + ["recording", "recording", "stages", "pack"])
        most = 4096 if kind == "layer" else 2048
        rows = int(round(math.exp(rng.uniform(0.0 if kind == "layer" else math.log(64), math.log(most)))))
        experts = int(round(math.exp(rng.uniform(math.log(8), math.log(512)))))
        inter = 128 * rng.randint(2, 8)
        shape = dict(d=256 * rng.randint(2, 10), experts=experts, topk=rng.randint(1, min(10, experts)), inter=inter,
                     shared=inter if rng.random() < 0.35 else 0)
        act, hc, skew = "f16", 0, False
        if kind == "layer":
            act, hc, skew = rng.choice([("f16", 0), ("f16", 0), ("f32", 4)]) + (rng.random() < 0.25,)
        elif kind == "recording":
            act, hc, skew = "f32", 4, rng.random() < 0.25
        elif kind == "stages":
            hc = rng.choice([0, 4])
        case = _case(kind, rows, shape, act=act, hc=hc, skew=skew)
        w = work(case)
        if w["bytes"] <= 5.2e9 and w["flops"] <= 2.6e11 and _weight_bytes(case) <= 5.1e9:
            return case


def _shape(case):
    return {k: case[k] for k in ("rows", "d", "experts", "topk", "inter", "shared")}


def _cols(case):
    return case["experts"] + (1 if case["shared"] else 0)


def _mrows(case):
    """Rows of the stages' expert-sorted buffers: every expert's segment padded to whole tiles."""
    return (case["rows"] * case["topk"] + case["experts"] * (TILE - 1) + TILE - 1) // TILE * TILE


def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _normal(g, shape, std=1.0, dtype=torch.float16):
    return torch.empty(shape, dtype=dtype, device="cuda").normal_(0.0, std, generator=g)


def _rank_bias(experts, rank):
    """A Zipf-like router bias: 3 log(1 / rank^1.2)."""
    return -3.6 * torch.log(rank[:experts].float())


def _weights(case, g, dtype=torch.float16):
    E, I, S, d = case["experts"], case["inter"], case["shared"], case["d"]
    w = {"w_router": _normal(g, (_cols(case), d), W_STD, torch.float32),
         "w_gate_up": _normal(g, (E, 2 * I, d), W_STD, dtype),
         "w_down": _normal(g, (E, d, I), W_STD, dtype),
         "w_sh_gate_up": None, "w_sh_down": None, "bias": None}
    if S:
        w["w_sh_gate_up"] = _normal(g, (2 * S, d), W_STD, dtype)
        w["w_sh_down"] = _normal(g, (d, S), W_STD, dtype)
    if case["skew"]:
        w["bias"] = _rank_bias(E, torch.randperm(E, generator=g, device="cuda") + 1)
    return w


def _streams(case, g):
    h = _normal(g, (case["rows"], case["hc"], case["d"]), 1.0, torch.float32)
    return h, _normal(g, (case["rows"], INJ_STRIDE), 3.0, torch.float32)


def _inputs(case, seed):
    """The inputs of a case, from the seed alone."""
    g = _gen(seed)
    E, T, K, d = case["experts"], case["rows"], case["topk"], case["d"]
    if case["kind"] == "pack":
        return _weights(case, g, torch.bfloat16)
    if case["kind"] == "stages":
        i = {"proj": _normal(g, (T, _cols(case)), 1.0, torch.float32), "x": _normal(g, (T, d)),
             "y": _normal(g, (_mrows(case), d), 0.2, torch.float32), "sh": None}
        if case["shared"]:
            i["sh"] = _normal(g, (T, d), 0.2, torch.float32)
    else:
        i = _weights(case, g)
        if case["kind"] == "recording" and i["bias"] is not None:
            # the recording's router takes no bias: the skew comes from a component that all tokens share
            common = _normal(g, (d,), 1.0, torch.float32)
            i["w_router"][:E] += i["bias"][:, None] * common[None, :] / (2.0 * d)
            i["bias"] = None
            i["x"] = _normal(g, (T, d), 1.0, torch.float32) + 2.0 * common
        else:
            i["x"] = _normal(g, (T, d), 1.0, torch.float16 if case["act"] == "f16" else torch.float32)
    if case["hc"]:
        i["h"], i["inj"] = _streams(case, g)
    return i


def prepare(case, seed):
    """What a program holds before the call: the context, the loaded weights, the workspace, the activations."""
    i = _inputs(case, seed)
    T, d, E, K = case["rows"], case["d"], case["experts"], case["topk"]
    s = dict(i, case=case, ctx=api.Context(0), shape=_shape(case))
    if case["kind"] == "pack":
        s["packed"] = torch.zeros(api.packed_bytes(s["shape"]) // 2, dtype=torch.float16, device="cuda")
        return s
    if not case["hc"]:
        s["out"] = torch.empty(T, d, dtype=torch.float16, device="cuda")
    if case["kind"] == "layer":
        need = api.workspace_bytes_x32 if case["act"] == "f32" else api.workspace_bytes
        s["ws"] = torch.empty(need(s["shape"]), dtype=torch.uint8, device="cuda")
        s["packed"] = s["ctx"].pack_weights(s["shape"], i["w_router"], i["w_gate_up"], i["w_down"], i["w_sh_gate_up"],
                                            i["w_sh_down"])
        for k in ("w_gate_up", "w_down", "w_sh_gate_up", "w_sh_down"):
            del s[k]  # the packed copy is what stays resident
    elif case["kind"] == "recording":
        s["rec"] = api.QwenMoe(s["ctx"], s["shape"], i["w_router"], i["w_gate_up"], i["w_down"], i["w_sh_gate_up"],
                               i["w_sh_down"], hc=case["hc"], hc_rank=INJ_OFF, inj_stride=INJ_STRIDE)
    else:
        m, u = _mrows(case), dict(dtype=torch.int32, device="cuda")
        s.update(idx=torch.empty(T * K, **u), wt=torch.empty(T * K, dtype=torch.float32, device="cuda"),
                 count=torch.empty(E, **u), off=torch.empty(E, **u), tiles=torch.empty(m // TILE, **u),
                 fill=torch.empty(E, **u), slot=torch.empty(T * K, **u),
                 xp=torch.zeros(m, d, dtype=torch.float16, device="cuda"))
    torch.cuda.synchronize()
    return s


def run(s):
    case, ctx = s["case"], s["ctx"]
    T, d, E, K, hc = case["rows"], case["d"], case["experts"], case["topk"], case["hc"]
    if case["kind"] == "pack":
        ctx.pack_weights(s["shape"], s["w_router"], s["w_gate_up"], s["w_down"], s["w_sh_gate_up"], s["w_sh_down"],
                         bf16=True, packed=s["packed"])
        return {"packed": s["packed"].view(torch.int16)}
    if case["kind"] == "layer":
        x, x32 = (s["x"], None) if case["act"] == "f16" else (None, s["x"])
        more = dict(h=s["h"], inj=s["inj"], inj_stride=INJ_STRIDE, inj_off=INJ_OFF, hc=hc) if hc else {}
        ctx.layer(s["shape"], x, s["w_router"], s["bias"], None, None, None, None, s.get("out"), s["ws"],
                  packed=s["packed"], x32=x32, **more)
        return {"h": s["h"]} if hc else {"out": s["out"]}
    if case["kind"] == "recording":
        s["rec"].moe_rec(s["x"], T, inj=s["inj"], h=s["h"])
        return {"h": s["h"]}
    ctx.route(T, E, K, _cols(case), s["proj"], s["idx"], s["wt"], s["count"])
    ctx.scan(E, TILE, s["count"], s["off"], s["tiles"], s["tiles"].numel())
    ctx.scatter_experts(E)
    ctx.scatter(T, K, d // 8, s["idx"], s["off"], s["fill"], s["x"], s["xp"], s["slot"])
    fields = (T, d, K, _cols(case), E, INJ_STRIDE if hc else 0, INJ_OFF if hc else 0, hc)
    proj = s["proj"] if case["shared"] else None
    if hc:
        ctx.combine(fields, s["wt"], s["slot"], s["y"], proj, s["sh"], s["inj"], s["h"])
    else:
        ctx.combine_plain(fields, s["wt"], s["slot"], s["y"], proj, s["sh"], s["out"])
    got = {k: s[k] for k in ("idx", "wt", "count", "off", "tiles", "slot", "xp")}
    got["h" if hc else "out"] = s["h"] if hc else s["out"]
    return got


def _touched(case):
    """Experts that a call's tokens reach, from a draw of the same logits on the CPU."""
    r = np.random.default_rng(0)
    rows = min(case["rows"], 1024)
    z = r.standard_normal((rows, case["experts"]), dtype=np.float32) * (W_STD * math.sqrt(case["d"]))
    if case["skew"]:
        z += np.float32(-3.6) * np.log(np.arange(1, case["experts"] + 1, dtype=np.float32))
    k = case["topk"]
    return len(np.unique(np.argpartition(-z, k - 1, axis=1)[:, :k])) if k < case["experts"] else case["experts"]


def _weight_bytes(case):
    return 6 * case["d"] * (case["experts"] * case["inter"] + case["shared"])


def work(case):
    T, d, E, K, I, S, hc = (case[k] for k in ("rows", "d", "experts", "topk", "inter", "shared", "hc"))
    router = _cols(case) * d * 4
    if case["kind"] == "pack":
        return {"bytes": 2.0 * (_weight_bytes(case) + router), "flops": 0.0}
    ends = T * d * (8 * hc if hc else 2) + (T * hc * 4 if hc else 0)  # the streams are read and written
    if case["kind"] == "stages":
        pairs = T * K * (3 * 4) + T * _cols(case) * 4
        return {"bytes": float(pairs + T * d * 2 + T * K * d * 2 + T * K * d * 4 + (T * d * 4 if S else 0) + ends),
                "flops": 2.0 * T * K * d}
    act = T * d * (2 if case["act"] == "f16" else 4)
    experts = 6 * d * (_touched(case) * I + S)
    return {"bytes": float(experts + router + act + ends),
            "flops": 6.0 * T * d * (K * I + S) + 2.0 * T * d * _cols(case)}


def tolerance(case):
    if case["kind"] == "pack":
        return "exact"
    if case["kind"] == "stages":
        # sums of at most ten fp32 products; the plain output is rounded to fp16
        return {"rel": 1e-6 if case["hc"] else 1e-3}
    # about four times what fp16 outputs, SwiGLU values and expert rows show against 64 bits (3.6e-4 of the layer's own
    # output); in the streams that share is smaller by what the output is added to, least where one expert dominates
    if case["hc"]:
        return {"rel": 2.5e-4 if case["topk"] >= 4 and not case["skew"] else 6e-4}
    return {"rel": 1.5e-3}


def _slot_cast(x):
    """x as the slot-scaled cast holds it: fp16 after a power of two that puts the largest magnitude in 2^14..2^15."""
    _, e = torch.frexp(x.abs().max())
    scale = 2.0 ** (15 - int(e))
    return (x * scale).half().double() / scale


def _gate(inj, hc):
    return 2.0 * torch.sigmoid(inj[:, INJ_OFF:INJ_OFF + hc].double() / hc)


def _ffn(x, gate_up, down):
    g, u = (x @ gate_up.double().T).chunk(2, dim=1)
    return (torch.nn.functional.silu(g) * u) @ down.double().T


def exact(case, seed):
    if case["kind"] == "pack":
        return None
    i = _inputs(case, seed)
    T, E, K, d, hc = case["rows"], case["experts"], case["topk"], case["d"], case["hc"]
    if case["kind"] == "stages":
        logits = i["proj"].double()
    else:
        x = i["x"].double() if case["act"] == "f16" else _slot_cast(i["x"])
        logits = x @ i["w_router"].double().T
        if i["bias"] is not None:
            logits[:, :E] += i["bias"].double()
    top, idx = torch.topk(logits[:, :E], K, dim=1)
    wt = torch.softmax(top, dim=1)
    y = torch.zeros(T, d, dtype=torch.float64, device="cuda")
    if case["kind"] == "stages":
        pair = idx.reshape(-1)
        count = torch.bincount(pair, minlength=E)
        padded = (count + TILE - 1) // TILE * TILE
        off = torch.cumsum(padded, 0) - padded
        order = torch.sort(pair, stable=True).indices
        slot = torch.empty_like(pair)
        first = torch.cumsum(count, 0) - count
        slot[order] = off[pair[order]] + torch.arange(T * K, device="cuda") - first[pair[order]]
        for j in range(K):
            y += wt[:, j, None] * i["y"][slot.view(T, K)[:, j]].double()
        if case["shared"]:
            y += torch.sigmoid(logits[:, E, None]) * i["sh"].double()
    else:
        for e in range(E):
            row, j = torch.nonzero(idx == e, as_tuple=True)
            if row.numel():
                y.index_add_(0, row, wt[row, j, None] * _ffn(x[row], i["w_gate_up"][e], i["w_down"][e]))
        if case["shared"]:
            y += torch.sigmoid(logits[:, E, None]) * _ffn(x, i["w_sh_gate_up"], i["w_sh_down"])
    end = {"h": i["h"].double() + y[:, None, :] * _gate(i["inj"], hc)[:, :, None]} if hc else {"out": y}
    if case["kind"] == "stages":
        end.update(idx=None, wt=wt.reshape(-1), count=None, off=None, tiles=None, slot=None, xp=None)
    return end
