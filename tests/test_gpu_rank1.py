"""The one-workgroup rank launch (calls of at most 1024 pairs with the
streaming tile's work list) against the oracle, bit for bit: counts, offsets,
slots and the selections, with the top-k folded in (up to 16 rows) and routed
by the router kernel, at its edges: one pair, 64-pair groups, 16 and 17 rows,
1024 pairs and the first call past them, 512 experts, experts without rows,
several items per expert and a shared group, and tokens nothing is selectable
for."""
import numpy as np
import pytest
import torch

from gpu_util import u32
from oracle import oracle as orc
from rmda_moe import api, inputs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,experts,topk,shared", [
    (1, 1, 1, 0), (1, 512, 16, 0), (8, 128, 8, 0), (9, 40, 7, 128), (16, 512, 10, 128), (16, 100, 16, 0),
    (17, 100, 3, 0), (64, 16, 16, 128), (65, 16, 16, 0), (1024, 2, 1, 0), (700, 3, 1, 128), (1025, 8, 1, 0),
])
def test_rank1_matches_oracle(rows, experts, topk, shared):
    torch.cuda.set_device(0)
    ctx = api.Context(0)
    cfg = dict(name="rank1", rows=rows, d=256, experts=experts, topk=topk, inter=128, shared=shared, skew=experts > 30)
    inp = inputs.make_inputs(ctx, cfg, seed=rows)
    if rows > 8:
        inp["x"][rows // 2] = float("nan")  # every logit NaN: no expert
    shape = inp["shape"]
    packed = ctx.pack_weights(shape, inp["w_router"], inp["w_gate_up"], inp["w_down"], inp["w_sh_gate_up"],
                              inp["w_sh_down"])
    ws = torch.full((api.workspace_bytes(shape),), 255, dtype=torch.uint8, device="cuda")
    out = torch.empty(rows, 256, dtype=torch.float16, device="cuda")
    ctx.layer(shape, inp["x"], inp["w_router"], inp["bias"], None, None, None, None, out, ws, packed=packed)
    ctx.sync()
    v = api.ws_views(shape, ws)
    ref = orc.layer(inputs.to_host(inp), tile=16, threads=16)
    for k in ("idx", "count", "off", "slot"):
        assert np.array_equal(u32(v[k]), ref[k]), k
    n = int(u32(v["n_items"])[0]) + int(u32(v["n_items_hot"])[0])
    lay = api.workspace_layout(shape)
    items = ws[lay["items"]:lay["items"] + 16 * n].view(torch.int32).view(n, 4).cpu().numpy()
    got = {}
    for e, row0, r, _ in items:
        got.setdefault(int(e), []).append((int(row0), int(r)))
    for e in range(experts):  # an expert's items tile its rows
        at = int(ref["off"][e])
        for row0, r in sorted(got.pop(e, [])):
            assert row0 == at and r > 0
            at += r
        assert at == int(ref["off"][e]) + int(ref["count"][e])
    assert sum(r for _, r in got.pop(experts, [])) == (rows if shared else 0) and not got
    ctx.close()
