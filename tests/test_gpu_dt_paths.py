"""The dt reduction with the blocks' maxima reduced on the host (up to 1024
blocks, no kernel sets the small-value flag) against the reduction kernel
(more blocks, or a configuration that may set the flag), and both against the
oracle, bit for bit; NaN cells are passed over by both."""
from __future__ import annotations

import numpy as np
import pytest

from amrvac_amd import problems
from amrvac_amd.host import Par
from amrvac_amd.mesh import UniformMesh

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny", [(16, 16), (80, 48), (512, 512), (528, 512)])
@pytest.mark.parametrize("bound", ["Einfeldt", "cmaxmean"])
@pytest.mark.parametrize("nan", [False, True])
def test_dt_of_both_reductions_matches_oracle(nx, ny, bound, nan):
    from amrvac_amd.fv import DeviceFV
    from oracle.oracle import OracleFV
    print(f"[dt] {nx} x {ny} {bound} nan {nan}", flush=True)
    par = Par(physics="hd", ndim=2, ndir=2, gamma=1.4, typeboundspeed=bound, flux_scheme="hll", limiter="minmod",
              courantpar=0.4)
    mesh = UniformMesh(2, (nx, ny), (16, 16), (0.0, 0.0), (nx / 16.0, ny / 16.0), ("periodic",) * 4, nghost=par.nghost)
    rng = np.random.default_rng(nx + ny)
    w = np.empty((mesh.nblocks, 4) + mesh.nxg[::-1])
    w[:, 0] = rng.uniform(0.5, 2.0, w[:, 0].shape)
    w[:, 1] = rng.uniform(-1.0, 1.0, w[:, 0].shape)
    w[:, 2] = rng.uniform(-1.0, 1.0, w[:, 0].shape)
    w[:, 3] = rng.uniform(5.0, 9.0, w[:, 0].shape)
    be = DeviceFV(par, mesh, precision="fp64")
    assert be.may_flag_small == (bound == "cmaxmean")
    be.set_state(0, w)
    orc = OracleFV(par, mesh, threads=2)
    orc.set_state(0, w)
    want = orc.getdt_courant(0, par.courantpar)
    assert be.getdt_courant(0, par.courantpar) == want
    assert not be.crash()
    if nan:
        # a NaN in a cell that does not hold the maximum changes nothing
        v = mesh.interior(w)
        speed = np.abs(v[:, 1] / v[:, 0]) + np.abs(v[:, 2] / v[:, 0])
        b, j, i = np.unravel_index(np.argmin(speed), speed.shape)
        v[b, 3, j, i] = np.nan
        be.set_state(0, w)
        assert be.getdt_courant(0, par.courantpar) == want
