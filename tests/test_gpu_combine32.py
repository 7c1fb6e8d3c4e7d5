"""The drop-in combine against the oracle at its kernel's edges: widths that
fill part of a wave (4, 260, 1024 columns), top-k around the read-ahead of 8
rows and the top-1 and top-2 variant, 1 to 8 streams around the 4 read ahead,
one and several waves per workgroup, pairs without a slot.  Both sides add the
same fp32 terms in the same order; a fused multiply-add on one side only moves
a term by half an ulp of it, 17 terms and 3 roundings of a stream at most."""
import numpy as np
import pytest
import torch

from gpu_util import dev
from oracle import oracle as orc
from rmda_moe import api

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,d,topk,shared,hc", [
    (1, 4, 1, False, 1), (3, 260, 2, True, 4), (5, 1024, 7, False, 5), (9, 512, 8, True, 8), (40, 256, 9, False, 4),
    (65, 2048, 16, True, 3), (1100, 256, 1, False, 4), (1100, 512, 3, True, 6),
])
def test_combine_edges(rows, d, topk, shared, hc):
    torch.cuda.set_device(0)
    ctx = api.Context(0)
    r = np.random.default_rng(rows * d + topk)
    n = rows * topk + 5
    slot = r.permutation(n)[:rows * topk].astype(np.uint32)
    if rows > 1:
        slot[r.integers(0, rows * topk, 3)] = 0xFFFFFFFF
    wt = r.random(rows * topk).astype(np.float32)
    y = r.standard_normal((n, d)).astype(np.float32)
    p = r.standard_normal((rows, 3)).astype(np.float32)
    sh = r.standard_normal((rows, d)).astype(np.float32) if shared else None
    inj = r.standard_normal((rows, hc + 2)).astype(np.float32)
    h0 = r.standard_normal((rows, hc, d)).astype(np.float32)
    fields = (rows, d, topk, 3, 2, hc + 2, 1, hc)
    want = orc.combine(fields, wt, slot, y, p, sh, inj, h0).reshape(rows, hc, d)
    h = dev(h0)
    args = (dev(wt), dev(slot), dev(y), dev(p), None if sh is None else dev(sh))
    ctx.combine(fields, *args, dev(inj), h)
    out = torch.empty(rows, d, dtype=torch.float16, device="cuda")
    ctx.combine_plain(fields, *args, out)
    ctx.sync()
    terms = np.zeros((rows, d))
    for j in range(topk):
        s = slot.reshape(rows, topk)[:, j]
        live = s != 0xFFFFFFFF
        terms[live] += wt.reshape(rows, topk)[live, j, None] * np.abs(y[s[live]].astype(np.float64))
    if shared:
        terms += np.abs(sh)
    eps = 2.0 ** -24
    gap = np.abs(h.cpu().numpy().astype(np.float64) - want)
    assert (gap <= eps * (2 * 17 * terms[:, None, :] + 3 * np.abs(want) + 3 * np.abs(h0) + 1e-30)).all()
    acc = orc.combine_plain(fields, wt, slot, y, p, sh)
    acc = np.asarray(acc).view(np.float16) if np.asarray(acc).dtype == np.uint16 else np.asarray(acc)
    gap = np.abs(out.float().cpu().numpy().astype(np.float64) - acc.astype(np.float64).reshape(rows, d))
    assert (gap <= 2.0 ** -10 * np.abs(acc.astype(np.float64).reshape(rows, d)) + 2 * 17 * eps * terms + 2.0 ** -24).all()
    ctx.close()
