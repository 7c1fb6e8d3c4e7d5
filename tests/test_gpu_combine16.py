"""The fused layer's combine at its edges: columns that fill part of a wave
(hidden 256, 768, 1280), top-k around the read-ahead of 8 rows and its top-1
and top-2 variant, 1 to 8 streams around the 4 read ahead, both outputs
together, one and several waves per workgroup, and tokens no expert was
selectable for.  The expected values are the layer's own expert rows summed in
float64 from the workspace's slots and weights; fp16 outputs may differ by one
rounding, the fp32 streams by the rounding of at most 17 terms."""
import numpy as np
import pytest
import torch

from rmda_moe import api, inputs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,d,experts,topk,shared,hc,with_out", [
    (1, 256, 4, 1, 0, 0, True), (5, 768, 8, 2, 128, 1, True), (7, 1280, 12, 7, 0, 3, False),
    (33, 512, 16, 8, 128, 4, True), (9, 256, 16, 9, 0, 5, True), (300, 2048, 16, 16, 128, 8, False),
    (1100, 512, 3, 1, 0, 0, True), (1100, 256, 5, 3, 128, 2, True),
])
def test_combine_against_expert_rows(rows, d, experts, topk, shared, hc, with_out):
    torch.cuda.set_device(0)
    ctx = api.Context(0)
    cfg = dict(name="comb", rows=rows, d=d, experts=experts, topk=topk, inter=128, shared=shared, skew=False)
    inp = inputs.make_inputs(ctx, cfg, seed=rows + d)
    if rows > 4:
        inp["x"][3] = float("nan")
    shape = inp["shape"]
    packed = ctx.pack_weights(shape, inp["w_router"], inp["w_gate_up"], inp["w_down"], inp["w_sh_gate_up"],
                              inp["w_sh_down"])
    ws = torch.zeros(api.workspace_bytes(shape), dtype=torch.uint8, device="cuda")
    g = torch.Generator(device="cuda").manual_seed(1)
    out = torch.zeros(rows, d, dtype=torch.float16, device="cuda") if with_out else None
    more, h0 = {}, None
    if hc:
        h0 = torch.randn(rows, hc, d, device="cuda", generator=g)
        more = dict(h=h0.clone(), inj=torch.randn(rows, hc + 3, device="cuda", generator=g), inj_stride=hc + 3,
                    inj_off=2, hc=hc)
    ctx.layer(shape, inp["x"], inp["w_router"], inp["bias"], None, None, None, None, out, ws, packed=packed, **more)
    ctx.sync()
    v = api.ws_views(shape, ws)
    slot = v["slot"].view(rows, topk).long() & 0xFFFFFFFF
    sh_row0 = (rows * topk + experts * 15 + 15) // 16 * 16
    groups = sh_row0 + ((rows + 15) // 16 * 16 if shared else 0)
    ye = ws[-((groups * d * 2 + 255) // 256 * 256):][:groups * d * 2].view(torch.float16).view(groups, d).double()
    want = torch.zeros(rows, d, dtype=torch.float64, device="cuda")
    size = torch.zeros_like(want)
    wt = v["wt"].view(rows, topk).double()
    for j in range(topk):
        live = slot[:, j] != 0xFFFFFFFF
        term = torch.zeros_like(want)
        term[live] = wt[live, j, None] * ye[slot[live, j]]
        want += term
        size += term.abs()
    if shared:
        term = torch.sigmoid(v["proj"][:, experts].double())[:, None] * ye[sh_row0:sh_row0 + rows]
        want += term
        size += term.abs()
    fine = torch.isfinite(want).all(dim=1)
    assert int(fine.sum()) >= rows - 1
    if with_out:
        bound = 2.0 ** -11 * want.abs() + 2.0 ** -22 * size * 17 + 2.0 ** -25
        assert ((out.double() - want).abs() <= bound)[fine].all()
    if hc:
        gate = 2.0 * torch.sigmoid(more["inj"][:, 2:2 + hc].double() / hc)
        ref = h0.double() + want[:, None, :] * gate[:, :, None]
        bound = 2.0 ** -22 * (17 * size[:, None, :] * gate[:, :, None] + ref.abs() + h0.double().abs())
        assert ((more["h"].double() - ref).abs() <= bound)[fine].all()
    assert np.isfinite(float(want[fine].abs().max()))
    ctx.close()
