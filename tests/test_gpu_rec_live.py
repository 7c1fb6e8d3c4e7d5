"""The recording's routed GEMMs, whose work items are up to 128 or up to 192
rows of an expert by what saves rounds of tasks, against the public grouped
GEMM over 128-row tiles: hp and its slot on every row that holds a routed pair,
and what the combine makes of ye, bitwise equal.  One expert with all rows gives exact counts on both sides
of an item's edge (4096 rows: 128-row items in gate_up, 192 in down; 4097 and
4224: 192 in both, a last item of 65 rows and none; 192 rows: one round either
way); the others have ragged and skewed experts, and 512 experts with so many
rows that the item list is too small for them and the 128-row tiles run."""
import numpy as np
import pytest
import torch

from gpu_util import u32
from rmda_moe import api, inputs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,d,experts,topk,inter,skew", [
    (192, 512, 1, 1, 256, False), (4096, 2560, 1, 1, 1024, False), (4097, 2560, 1, 1, 1024, False),
    (4224, 2560, 1, 1, 1024, False), (2048, 2560, 16, 2, 1024, False), (1700, 1024, 128, 8, 768, False),
    (2048, 512, 128, 8, 256, True), (12400, 256, 512, 16, 128, False),
])
def test_live_rows_bitwise(rows, d, experts, topk, inter, skew):
    print("rec live", rows, d, experts, topk, inter, skew, flush=True)
    torch.cuda.set_device(0)
    ctx = api.Context(0)
    cfg = dict(name="rec", rows=rows, d=d, experts=experts, topk=topk, inter=inter, shared=0, skew=skew)
    inp = inputs.make_inputs(ctx, cfg, seed=rows)
    q = api.QwenMoe(ctx, inp["shape"], inp["w_router"], inp["w_gate_up"], inp["w_down"], None, None)
    q.scratch.fill_(255)
    out = torch.empty(rows, d, dtype=torch.float16, device="cuda")
    q.moe_rec(inp["x"].float(), rows, out=out)
    ctx.sync()
    v = q.views(rows)
    m = v["hp"].shape[0]
    live = torch.zeros(m, dtype=torch.bool, device="cuda")
    for o, c in zip(u32(v["off"]), u32(v["count"])):
        live[int(o):int(o) + int(c)] = True
    assert live.sum().item() == rows * topk
    slots = v["amax"].clone()
    lay = q.layout
    xp = q.scratch[lay["xp"]:lay["xp"] + m * d * 2].view(torch.float16).view(m, d)
    g = torch.empty(m, 2 * inter, device="cuda")
    ctx.mm(m, 2 * inter, d, 0, 0xFFFFFFFF, xp, inp["w_gate_up"], g, slots, v["tiles"])
    hp = torch.empty(m, inter, device="cuda")
    ctx.qwen_elem(m, inter, 2 * inter, 0, inter, 0, 1.0, g, hp)
    ye = torch.empty(m, d, device="cuda")
    ctx.mm(m, d, inter, 1, 0xFFFFFFFF, v["hp16"], inp["w_down"], ye, slots, v["tiles"])
    want = torch.empty_like(out)
    ctx.combine_plain((rows, d, topk, v["p"].shape[1], experts, 0, 0, 0), v["wt"], v["slot"], ye, v["p"], None, want)
    ctx.sync()
    bits = lambda t: t.contiguous().view(torch.int32)[live]  # noqa: E731
    assert torch.isfinite(hp[live]).all()
    assert torch.equal(bits(v["hp"]), bits(hp))
    amax = np.float32(hp[live].abs().max().item())
    assert slots[1].item() == int(amax.view(np.int32))
    assert torch.equal(out.view(torch.int16), want.view(torch.int16))
    ctx.close()
