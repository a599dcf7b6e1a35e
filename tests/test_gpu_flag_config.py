"""Which configurations may raise the small-value flag: the host's rule and the
flag itself, on a state whose pressure is below small_pressure (HD cmaxmean
raises it; the other bounds and MHD leave it as it is).  On more than 1024
blocks the dt reduction reads the flag itself."""
from __future__ import annotations

import numpy as np
import pytest

from amrvac_amd.host import FS, Par
from amrvac_amd.mesh import UniformMesh

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("physics", ["hd", "mhd"])
@pytest.mark.parametrize("bound", ["Einfeldt", "cmaxmean", "cmaxleftright"])
def test_flag_is_raised_only_where_the_rule_says(physics, bound):
    from amrvac_amd.fv import DeviceFV
    print(f"[flag] {physics} {bound}", flush=True)
    par = Par(physics=physics, ndim=2, ndir=2 if physics == "hd" else 3, gamma=1.4, typeboundspeed=bound,
              flux_scheme="hll", limiter="minmod", small_pressure=1.0)
    mesh = UniformMesh(2, (528, 512), (16, 16), (0.0, 0.0), (33.0, 32.0), ("periodic",) * 4, nghost=par.nghost)
    assert mesh.nblocks > 1024
    w = np.zeros((mesh.nblocks, par.nw) + mesh.nxg[::-1])
    w[:, 0] = 1.0
    e = par.ndir + 1
    w[:, e] = 0.5 / 0.4  # p = 0.5 < small_pressure
    be = DeviceFV(par, mesh, precision="fp64")
    be.set_state(0, w)
    dt, ch = be.getdt_courant(0, 0.4)
    be.advect1(FS["hll"], 1.0, dt, ch, 0, 1, ("copy", 0))
    be.getdt_courant(1, 0.4)
    assert be.may_flag_small == (physics == "hd" and bound == "cmaxmean")
    assert be.crash() == be.may_flag_small
