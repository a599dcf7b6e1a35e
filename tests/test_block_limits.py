"""A block whose variables do not fit 32-bit byte offsets is refused when the
context is made (no GPU needed: the check comes before the device is touched)."""
from __future__ import annotations

import ctypes
import os

import pytest

from amrvac_amd import fv


@pytest.mark.parametrize("physics,divb,planes", [(1, 0, 419430), (2, 0, 262143), (2, 1, 233016)])
def test_block_of_4_gib_is_refused(physics, divb, planes):
    """planes: the most of a 16^2 cross-section that fit (5, 8 and 9 variables)."""
    if not os.path.exists(fv.LIB_PATH):
        pytest.skip("library not built")
    L = fv.load_library()
    cfg = fv.FVConfig()
    cfg.ndim, cfg.ndir, cfg.physics, cfg.gamma, cfg.divb = 3, 3, physics, 1.4, divb
    cfg.limiter, cfg.boundspeed, cfg.nghost, cfg.precision = 5, 1, 2, 0
    for n, refused in ((planes, False), (planes + 1, True), (2147483647, True)):
        cfg.block_nx[0], cfg.block_nx[1], cfg.block_nx[2] = 16, 16, n
        h = ctypes.c_void_p()
        rc = L.amrvac_fv_init(ctypes.byref(cfg), ctypes.byref(h))
        assert (rc == -1 and b"4 GiB" in L.amrvac_fv_last_error()) == refused
        if rc == 0:
            L.amrvac_fv_finalize(h)
