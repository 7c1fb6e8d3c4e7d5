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
