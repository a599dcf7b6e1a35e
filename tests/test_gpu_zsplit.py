"""3-D stages whose blocks' planes are split over several workgroups (levels
with few blocks): the contraction-free kernels against the oracle bit for bit
at depths that split into parts of 4 to 10 planes or not at all, and the mixed
form's fused CFL partials (one pair per workgroup) against the separate pass."""
from __future__ import annotations

import numpy as np
import pytest

from amrvac_amd import problems
from amrvac_amd.host import Par, TimeIntegrator
from amrvac_amd.mesh import UniformMesh

pytestmark = pytest.mark.gpu


def _setup(bz, nbz, bc, limiter="cada3", flux="hll", stepper="threestep"):
    par = Par(physics="mhd", ndim=3, ndir=3, gamma=5.0 / 3.0, typedivbfix="glm", flux_scheme=flux, limiter=limiter,
              typeboundspeed="Einfeldt", time_stepper=stepper, courantpar=0.5)
    nz = bz * nbz
    mesh = UniformMesh(3, (32, 16, nz), (16, 16, bz), (0.0,) * 3, (1.0, 0.5, nz / 32.0), bc, nghost=par.nghost)
    return par, mesh, problems.orszag_tang_3d(mesh)


@pytest.mark.parametrize("bz,nbz,limiter,flux,stepper", [
    (4, 2, "cada3", "hll", "threestep"), (8, 2, "vanleer", "hll", "threestep"), (12, 1, "cada3", "hll", "threestep"),
    (10, 2, "minmod", "tvdlf", "twostep"), (16, 1, "weno5", "hll", "threestep"), (20, 2, "koren", "hll", "threestep"),
    (18, 1, "cada3", "hlld", "threestep")])
def test_split_blocks_match_oracle_bitwise(bz, nbz, limiter, flux, stepper):
    from amrvac_amd.fv import DeviceFV
    from oracle.oracle import OracleFV
    print(f"[zsplit] {bz} x {nbz} {limiter} {flux}", flush=True)
    par, mesh, w0 = _setup(bz, nbz, ("periodic", "periodic", "cont", "cont", "symm", "cont"), limiter, flux, stepper)
    out = []
    for be in (OracleFV(par, mesh, threads=2), DeviceFV(par, mesh, precision="fp64_exact")):
        be.set_state(0, w0)
        be.getbc(0)
        ti = TimeIntegrator(par, mesh, be)
        ti.run(nsteps=2)
        out.append((mesh.interior(be.get_state(0)), ti.state.dts))
    assert out[1][1] == out[0][1]
    assert np.array_equal(out[1][0], out[0][0])


@pytest.mark.parametrize("bz,nbz", [(16, 1), (12, 2), (20, 1)])
def test_split_blocks_fused_dt(bz, nbz):
    from amrvac_amd.fv import DeviceFV
    print(f"[zsplit] fused dt {bz} x {nbz}", flush=True)
    par, mesh, w0 = _setup(bz, nbz, ("periodic",) * 6)
    be = DeviceFV(par, mesh, precision="mixed")
    be.set_state(0, w0)
    ti = TimeIntegrator(par, mesh, be)
    for _ in range(2):
        ti.step()
    fused = be.getdt_courant(0, par.courantpar)
    be.slot_pointer(0)  # the partials are dropped: the next call makes its own pass
    assert be.getdt_courant(0, par.courantpar) == fused
