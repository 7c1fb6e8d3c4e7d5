"""The strip GEMM of small calls (one wave per 64-row chunk and 32 weight rows)
against the streaming tile: the default policy takes the strip kernel at these
shapes, TILE_STREAM never does, and both run the same MFMA sequence per output
element, so the results are bitwise equal; the routing and output are also
held to the oracle's tolerance.  Which GEMMs take strips, with the deep ring of
K steps and walking the work list, is asserted per shape.  Shapes sit at the kernel's edges: one row, the
16-row groups and 64-row chunks (15..17, 63..65 rows on one expert), items of
192 rows, K loops shorter than, equal to and not a multiple of the ring, slabs
not a multiple of the 8 XCDs, a shared expert's rows in several chunks, and
launches of fewer waves than their bound on the tasks, each walking several,
with the chunks of an item in one wave and in several.
"""
import ctypes

import pytest
import torch

from gpu_util import MAX_ABS, REL_L2, f32, out_metrics
from oracle import oracle as orc
from rmda_moe import api, inputs
from test_cpu_rules import internal

pytestmark = pytest.mark.gpu


GU, DN = 1, 2  # bits: gate_up, down


def case(rows, d, experts, topk, inter, shared=False, skew=False, strips=GU | DN, deep=0, walk=0):
    return dict(name="strip", rows=rows, d=d, experts=experts, topk=topk, inter=inter,
                shared=inter if shared else 0, skew=skew), strips, deep, walk


CASES = [
    case(1, 256, 1, 1, 128),                      # K of 8 and 4 steps
    case(1, 2048, 128, 8, 768),                   # one token
    case(15, 512, 1, 1, 256), case(16, 512, 1, 1, 256), case(17, 512, 1, 1, 256),
    case(63, 768, 1, 1, 384), case(64, 768, 1, 1, 384), case(65, 768, 1, 1, 384, shared=True),
    case(200, 256, 2, 1, 128, shared=True),       # items of 192 rows and a remainder
    case(385, 256, 3, 2, 256, skew=True),
    case(33, 1024, 40, 6, 640, shared=True),      # 5 gate_up slabs
    case(37, 2304, 16, 3, 896),                   # 72 and 28 steps: not a multiple of 8 in down
    case(256, 512, 8, 2, 1024),
    case(16, 2560, 512, 10, 640, shared=True, deep=GU | DN),
    case(64, 1280, 300, 3, 512, skew=True, deep=GU | DN),  # most experts without rows
    # the deep ring (16, 12, 8 and 7 steps for 1 to 4 row groups) over 40 and 20 steps: the shared expert's 20, 40
    # and 60 rows are 2, 3 and 4 groups, the others' one
    case(20, 1280, 100, 8, 640, shared=True, deep=GU | DN), case(40, 1280, 100, 4, 640, shared=True, deep=GU | DN),
    case(60, 1280, 100, 2, 640, shared=True, deep=GU | DN),
    case(1, 768, 174, 1, 256),                    # fp32 activations: down casts the SwiGLU output
    case(3, 512, 182, 4, 256, shared=True), case(70, 512, 3, 1, 256), case(40, 512, 2, 2, 256, shared=True),
    # more tasks than waves: gate_up with an item's chunks in one wave, down split; few experts with rows
    case(180, 512, 512, 10, 384, shared=True, deep=GU, walk=GU | DN),
    case(180, 768, 512, 10, 384, skew=True, deep=GU, walk=GU | DN),
    case(1536, 512, 8, 2, 1024, strips=DN), case(975, 512, 13, 10, 384, strips=0),  # large experts
]


@pytest.fixture(scope="module")
def ctx():
    torch.cuda.set_device(0)
    c = api.Context(0)
    yield c
    c.close()


def run(ctx, inp, packed, policy, act, hc):
    shape = inp["shape"]
    T, d = shape["rows"], shape["d"]
    ctx.set_tile_policy(policy)
    need = api.workspace_bytes_x32 if act == "f32" else api.workspace_bytes
    ws = torch.full((need(shape),), 255, dtype=torch.uint8, device="cuda")  # NaN wherever nothing was written
    out = torch.full((T, d), float("nan"), dtype=torch.float16, device="cuda")
    more = {}
    if hc:
        more = dict(h=torch.zeros(T, hc, d, device="cuda"), inj=torch.ones(T, hc, device="cuda"), inj_stride=hc, hc=hc)
    x, x32 = (inp["x"], None) if act == "f16" else (None, inp["x"].float() * 1.001)
    ctx.layer(shape, x, inp["w_router"], inp["bias"], None, None, None, None, out, ws, packed=packed, x32=x32, **more)
    ctx.sync()
    ctx.set_tile_policy(api.Context.TILE_ADAPTIVE)
    return [out.view(torch.int16)] + ([more["h"].view(torch.int32)] if hc else [])


def chosen(cfg):
    """(strips, deep, walk) as the library decides them."""
    T, d, inter, sh = cfg["rows"], cfg["d"], cfg["inter"], cfg["rows"] if cfg["shared"] else 0
    strips = internal("rmda_gemm_strip_choice")(T, cfg["topk"], cfg["experts"], sh, inter, d)
    items = internal("rmda_gemm_strip_items")(T * cfg["topk"], cfg["experts"], sh)
    deep = walk = 0
    for bit, n_w, k in ((GU, 2 * inter, d), (DN, d, inter)):
        chunks = -(-min(T, 192) // 64)
        tasks = -(-items * (n_w // 256) // 8) * 8 * 8 * chunks
        if strips & bit:
            deep |= bit if internal("rmda_gemm_strip_deep", ctypes.c_bool)(items, n_w, k) else 0
            walk |= bit if internal("rmda_gemm_strip_waves")(items, min(T, 192), n_w) < tasks else 0
    return strips, deep, walk


@pytest.mark.parametrize("cfg,strips,deep,walk", CASES, ids=lambda c: "T%d-d%d-E%d-k%d-I%d-S%d" % (
    c["rows"], c["d"], c["experts"], c["topk"], c["inter"], c["shared"]) if isinstance(c, dict) else "%d" % c)
def test_strip_bitwise_and_oracle(ctx, cfg, strips, deep, walk):
    assert chosen(cfg) == (strips, deep, walk)
    inp = inputs.make_inputs(ctx, cfg, seed=3)
    packed = ctx.pack_weights(inp["shape"], inp["w_router"], inp["w_gate_up"], inp["w_down"], inp["w_sh_gate_up"],
                              inp["w_sh_down"])
    for act, hc in (("f16", 0), ("f16", 4), ("f32", 2)):
        got = run(ctx, inp, packed, api.Context.TILE_ADAPTIVE, act, hc)
        ref = run(ctx, inp, packed, api.Context.TILE_STREAM, act, hc)
        for g, r in zip(got, ref):
            assert torch.equal(g, r), (act, hc)
    if cfg["experts"] * cfg["d"] * cfg["inter"] <= 1 << 25:
        out = run(ctx, inp, packed, api.Context.TILE_ADAPTIVE, "f16", 0)[0]
        want = orc.layer(inputs.to_host(inp), tile=16, threads=16)["out"]
        max_abs, rel = out_metrics(f32(out.view(torch.float16)), want)
        assert max_abs <= MAX_ABS and rel <= REL_L2
