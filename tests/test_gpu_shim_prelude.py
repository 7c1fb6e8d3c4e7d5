"""The recording's merged launches (absmax, cast, router packing, cleared slots
and the shared expert's tile map in one or two; counts, offsets and tile map in
one) against the same recording with a 4-byte aligned x, which takes the stage
by stage launches: bitwise equal outputs, slots, counts, offsets, tile map and
slot words, at the sizes where the launches change (one-launch cast up to 49152
values, rows around the 128-row tiles, one and 512 experts).  x is finite with
its largest magnitude first, in the middle and last, so that slot 0 shows
whether every part of x was folded, and once holds an infinity."""
import pytest
import torch

from rmda_moe import api, inputs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,d,experts,topk,inter,shared", [
    (1, 256, 1, 1, 128, 0), (127, 256, 8, 2, 128, 128), (192, 256, 5, 3, 128, 0), (193, 256, 512, 10, 128, 128),
    (129, 512, 40, 7, 256, 256), (300, 768, 16, 16, 128, 384),
])
def test_prelude_bitwise(rows, d, experts, topk, inter, shared):
    torch.cuda.set_device(0)
    ctx = api.Context(0)
    cfg = dict(name="rec", rows=rows, d=d, experts=experts, topk=topk, inter=inter, shared=shared, skew=False)
    inp = inputs.make_inputs(ctx, cfg, seed=rows)
    g = torch.Generator(device="cuda").manual_seed(rows)
    base = torch.randn(rows * d, device="cuda", generator=g)
    if rows > 3:
        base[:d] *= 0.0
    q = api.QwenMoe(ctx, inp["shape"], inp["w_router"], inp["w_gate_up"], inp["w_down"], inp["w_sh_gate_up"],
                    inp["w_sh_down"])
    shifted = torch.empty(rows * d + 1, device="cuda")[1:]
    big = [(0, -97.5), (rows * d // 2 + 1, 3.0e5), (rows * d - 1, -1310.75)]
    for at, value in big + ([(3 * d + 1, float("inf"))] if rows > 3 else []):
        x = base.clone()
        x[at] = value
        shifted.copy_(x)
        got = []
        for a in (x, shifted):
            q.scratch.fill_(85)
            out = torch.zeros(rows, d, dtype=torch.float16, device="cuda")
            q.moe_rec(a.view(rows, d), rows, out=out)
            ctx.sync()
            v = q.views(rows)
            got.append([out.view(torch.int16)] +
                       [v[k].clone() for k in ("idx", "count", "off", "slot", "tiles", "amax")] +
                       [v["wt"].view(torch.int32).clone(), v["p"].contiguous().view(torch.int32).clone()])
        for a, b in zip(*got):
            assert torch.equal(a, b), at
        assert got[0][6][0].item() == x.abs().max().view(torch.int32).item(), at
    ctx.close()
