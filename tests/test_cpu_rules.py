"""Host-side rules of the dispatch, called in the built library (no kernel is
launched): what a launch is sized for, and which kernel a shape takes.  The
functions are internal C++ ones, found by their mangled names."""
import ctypes
import re
import subprocess

import pytest

from rmda_moe import _lib


def internal(name, restype=ctypes.c_uint32):
    out = subprocess.run(["nm", "-D", "--defined-only", _lib.LIB_PATH], capture_output=True, text=True, check=True).stdout
    sym = re.findall(r" T (_Z%d%s\w*)$" % (len(name), name), out, re.M)
    assert len(sym) == 1, (name, sym)
    f = getattr(_lib.lib(), sym[0])
    f.restype = restype
    return f


@pytest.mark.parametrize("items,item_rows,n_w,waves", [
    (1, 1, 256, 64), (8, 64, 2048, 512), (128, 16, 1536, 6144), (512, 64, 2560, 40960), (522, 192, 256, 12672),
    # the bound on the tasks (every expert, three chunks each) is 62640 and 125280 here, and a call under skewed
    # routing fills 800 of them
    (522, 192, 1280, 16384), (522, 192, 2560, 16384),
])
def test_strip_launch_is_bounded(items, item_rows, n_w, waves):
    assert internal("rmda_gemm_strip_waves")(items, item_rows, n_w) == waves


GATE_UP, DOWN = 1, 2


def strips(rows, d, experts, topk, inter, shared=0):
    """Which GEMMs of the fused layer (packed weights, default policy) take the strip kernel."""
    return internal("rmda_gemm_strip_choice")(rows, topk, experts, rows if shared else 0, inter, d)


@pytest.mark.parametrize("shape,want", [
    # few rows per expert: strips, also under skewed routing
    ((1, 2048, 128, 8, 768), 3), ((16, 2560, 512, 10, 640, 640), 3), ((51, 2560, 512, 10, 640), 3),
    ((400, 1280, 300, 3, 640), 3), ((200, 1792, 480, 6, 512), 3), ((512, 2048, 512, 1, 512), 3),
    # as few on average, but all on the same experts they cost more there than they gain: 9 to 24% of the layer
    ((102, 2560, 512, 10, 640), 0), ((199, 2560, 512, 10, 640), 0), ((65, 2048, 256, 8, 768), 0),
    ((96, 2560, 160, 5, 1024), 0), ((64, 2048, 256, 16, 768), 0), ((64, 2048, 256, 8, 768), 3),
    # few experts: the rows on average decide, and how full a round their tasks are (layer 50 -> 54 us in strips)
    ((256, 768, 64, 8, 256), 3), ((400, 768, 64, 8, 256), DOWN), ((1792, 512, 32, 4, 256), 0),
    ((1792, 2048, 8, 1, 256), 3),
    ((256, 512, 8, 2, 1024), 3), ((1536, 512, 8, 2, 1024), DOWN), ((975, 512, 13, 10, 384), 0),
    ((2048, 2048, 128, 8, 768), 0), ((777, 2048, 128, 8, 768), 0),
])
def test_strip_choice(shape, want):
    assert strips(*shape) == want


@pytest.mark.parametrize("n128,n192,ntiles,pairs,want", [
    # 64 experts top-8, 2048 x 768 (6 gate_up tiles, 8 of down) at 1100, 1300, 1400, 1900, 2300, 2700 and 3500 tokens
    (112, 64, 6, 8800, True), (112, 64, 8, 8800, True), (128, 65, 8, 10400, False), (128, 72, 8, 11200, False),
    (134, 128, 6, 15200, True), (134, 128, 8, 15200, True), (191, 128, 6, 18400, True), (191, 128, 8, 18400, True),
    (193, 129, 6, 21600, False), (193, 129, 8, 21600, True), (256, 192, 6, 28000, False), (256, 192, 8, 28000, True),
    # equal rounds, and no items
    (128, 107, 6, 12800, False), (128, 107, 8, 12800, False), (16, 16, 10, 1400, False), (0, 0, 8, 0, False),
])
def test_recording_item_height(n128, n192, ntiles, pairs, want):
    """The measured faster height of the recording's work items, where it differs by 2 us or more."""
    assert internal("rmda_ref_live_tall", ctypes.c_bool)(n128, n192, ntiles, 256, pairs) == want
