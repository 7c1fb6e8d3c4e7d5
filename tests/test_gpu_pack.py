"""rmda_moe_pack_weights against a numpy restatement of the packed format
(include/rmda_moe.h, csrc/common.h): slab images, router rows, and the down
weights' row-sum bound, bit for bit, at the edges of the packing tiles (one
128-column tile of down, several; one 256-column tile of gate_up, several; one
expert; a shared expert), from fp16 and from bf16, with rows that hold
infinities and NaN left out of the bound.
"""
import numpy as np
import pytest
import torch

from gpu_util import u16
from rmda_moe import api

pytestmark = pytest.mark.gpu


def slab_image(w, swiglu, inter):
    """[n_w][k] fp16 bits -> the packed slab image of one expert."""
    n_w, k = w.shape
    out = np.empty((n_w * k // 8, 8), dtype=np.uint16)
    n = np.arange(256)
    units = w.reshape(n_w, k // 8, 8)
    for t in range(n_w // 256):
        if swiglu:
            c = t * 128 + n // 64 * 32 + n % 32
            row = np.where(n % 64 < 32, c, inter + c)
        else:
            row = t * 256 + n
        for ks in range(k // 32):
            for p in range(4):
                at = ((t * (k // 32) + ks) * 256 + n) * 4 + p
                out[at] = units[row, ks * 4 + (p ^ (n >> 1 & 3))]
    return out.reshape(-1)


def row_sums(image, n_w, k):
    """Sequential fp32 sums of |w| in packed order, two values at a time."""
    a = np.abs(image.view(np.float16).reshape(n_w // 256, k // 32, 256, 32).astype(np.float32))
    a = a.transpose(0, 2, 1, 3).reshape(n_w, k // 2, 2)
    s = np.zeros(n_w, np.float32)
    with np.errstate(over="ignore", invalid="ignore"):
        pair = a[:, :, 0] + a[:, :, 1]
        for i in range(k // 2):
            s = s + pair[:, i]
    return s[np.isfinite(s)]


@pytest.mark.parametrize("E,d,inter,shared", [(1, 256, 128, False), (3, 512, 384, True), (2, 768, 256, False),
                                              (5, 1280, 640, True)])
@pytest.mark.parametrize("bf16", [False, True])
def test_pack_format(E, d, inter, shared, bf16):
    torch.cuda.set_device(0)
    ctx = api.Context(0)
    g = torch.Generator(device="cuda").manual_seed(E * d + inter)
    dt = torch.bfloat16 if bf16 else torch.float16
    rnd = lambda *s: (torch.randn(*s, device="cuda", generator=g) * 0.3).to(dt)  # noqa: E731
    S = inter if shared else 0
    cols = E + (1 if shared else 0)
    wr = torch.randn(cols, d, device="cuda", generator=g)
    gu, dn = rnd(E, 2 * inter, d), rnd(E, d, inter)
    sgu, sdn = (rnd(2 * S, d), rnd(d, S)) if shared else (None, None)
    dn[0, 3] *= 50.0  # the largest finite row sum
    dn[0, 5, 7] = float("inf")
    dn[E - 1, d - 1, inter - 1] = float("nan")
    shape = dict(rows=4, d=d, experts=E, topk=1, inter=inter, shared=S)
    packed = torch.full((api.packed_bytes(shape) // 2,), -1.0, dtype=torch.float16, device="cuda")
    ctx.pack_weights(shape, wr, gu, dn, sgu, sdn, bf16=bf16, packed=packed)
    ctx.sync()
    got = u16(packed)
    half = lambda t: u16(t.float().half())  # noqa: E731  (round to nearest even, as the kernel converts)
    want = [slab_image(half(gu[e]), True, inter) for e in range(E)]
    down = [slab_image(half(dn[e]), False, inter) for e in range(E)]
    tail = [slab_image(half(sgu), True, inter), slab_image(half(sdn), False, inter)] if shared else []
    want = np.concatenate(want + down + tail)
    nan = np.isnan(want.view(np.float16))
    assert np.array_equal(got[:want.size][~nan], want[~nan])
    assert np.isnan(got[:want.size].view(np.float16)[nan]).all()
    cpad = (cols + 63) // 64 * 64
    rt = np.zeros((d // 16, cpad, 4, 4), np.float32)  # [k / 16][column][k % 4][k % 16 / 4]
    rt[:, :cols] = wr.cpu().numpy().reshape(cols, d // 16, 4, 4).transpose(1, 0, 3, 2)
    end = want.size + 2 * d * cpad
    assert np.array_equal(got[want.size:end].view(np.float32), rt.reshape(-1))
    bound = max(row_sums(m, d, inter).max() for m in down + tail[1:])
    words = got[end:].view(np.float32)
    assert words.size == 64 and words[0] == bound and not words[1:].any()
    ctx.close()
