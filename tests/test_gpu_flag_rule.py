"""The library's rule for which configurations may raise the small-value flag,
against the flag on the device: after a stage on a state whose pressure is below
small_pressure everywhere, it is up only where the rule says it may be.  The
flag itself is read back with the dt maxima of more than 1024 blocks, and on a
tree with the refinement flags."""
from __future__ import annotations

import numpy as np
import pytest

from amrvac_amd.amr import AMRForest, AMRPar
from amrvac_amd.fv import DeviceFV
from amrvac_amd.host import FS, Par
from amrvac_amd.mesh import UniformMesh

pytestmark = pytest.mark.gpu


def _par(physics, ndim, bound, limiter="minmod", **kw):
    return Par(physics=physics, ndim=ndim, ndir=ndim if physics == "hd" else 3, gamma=1.4, typeboundspeed=bound,
               flux_scheme="hll", limiter=limiter, small_pressure=1.0, **kw)


def _low_pressure(par, shape):
    w = np.zeros(shape)
    w[:, 0] = 1.0
    w[:, par.ndir + 1] = 0.5 / (par.gamma - 1.0)  # p = 0.5
    return w


# physics, ndim, flux, limiter, bound speeds, precision, options, block edge, may raise it, does raise it
UNIFORM = [
    ("hd", 2, "hllc", "vanleer", "cmaxmean", "mixed", {}, 16, True, True),
    ("hd", 2, "hancock", "minmod", "cmaxmean", "fp64", {}, 16, True, False),  # the predictor has no speeds
    ("hd", 2, "tvdlf", "weno5", "cmaxleftright", "fp64", {}, 16, False, False),
    ("hd", 2, "hll", "minmod", "cmaxmean", "fp64", dict(check_small_values=False), 16, False, False),
    ("hd", 2, "hll", "albada", "Einfeldt", "fp64", dict(fix_small_values=True), 16, True, True),
    ("mhd", 2, "hlld", "minmod", "cmaxmean", "fp64_exact", {}, 16, False, False),
    ("mhd", 2, "hll", "cada3", "cmaxmean", "mixed", dict(typedivbfix="glm"), 16, False, False),
    ("mhd", 2, "hll", "vanleer", "cmaxmean", "fp64", dict(typedivbfix="linde"), 16, False, False),
    ("mhd", 2, "hll", "cada3", "cmaxmean", "fp64", dict(typedivbfix="ct", type_ct="uct_contact"), 16, False, False),
    ("mhd", 2, "hancock", "minmod", "cmaxmean", "fp64", dict(typedivbfix="ct", type_ct="average"), 16, False, False),
    ("hd", 3, "tvdlf", "cada3", "cmaxmean", "fp64", {}, 8, True, True),
    ("mhd", 3, "hll", "weno5", "cmaxmean", "fp64", dict(typedivbfix="glm"), 8, False, False),
    ("mhd", 3, "hllc", "koren", "Einfeldt", "fp64", dict(typedivbfix="linde"), 10, False, False),
    ("mhd", 3, "hll", "vanleer", "cmaxmean", "mixed", dict(typedivbfix="glm"), 16, False, False),
    ("hd", 3, "hll", "vanleer", "Einfeldt", "fp64", {}, 16, False, False),
]


@pytest.mark.parametrize("physics,ndim,flux,limiter,bound,precision,options,edge,may,does", UNIFORM)
def test_flag_on_a_uniform_level(physics, ndim, flux, limiter, bound, precision, options, edge, may, does):
    print(f"[flag rule] {physics} {ndim}-D {flux} {limiter} {bound} {precision} {options}", flush=True)
    par = _par(physics, ndim, bound, limiter, **options)
    block = (edge, edge, 4)[:ndim]
    dims = (33 * edge, 32 * edge, 4)[:ndim]
    mesh = UniformMesh(ndim, dims, block, (0.0,) * ndim, tuple(float(n) for n in dims), ("periodic",) * (2 * ndim),
                       nghost=par.nghost)
    assert mesh.nblocks > 1024
    be = DeviceFV(par, mesh, precision=precision)
    be.set_state(0, _low_pressure(par, (mesh.nblocks, par.nwt) + mesh.nxg[::-1]))
    be.slot_pointer(0)  # dt comes from a pass of its own in every precision
    dt, ch = be.getdt_courant(0, 0.4)
    be.crash(clear=True)
    be.advect1(FS[flux], 1.0, dt, ch, 0, 1, ("copy", 0))
    be.getdt_courant(1, 0.4)
    assert be.may_flag_small == may
    assert be.crash() == does
    be.close()


@pytest.mark.parametrize("physics,bound,divb,may", [("hd", "cmaxmean", "none", True), ("hd", "Einfeldt", "none", False),
                                                    ("mhd", "cmaxmean", "linde", False),
                                                    ("mhd", "cmaxmean", "glm", False)])
@pytest.mark.parametrize("ndim", [2, 3])
def test_flag_on_a_tree(ndim, physics, bound, divb, may):
    print(f"[flag rule] tree {ndim}-D {physics} {bound} {divb}", flush=True)
    par = _par(physics, ndim, bound, typedivbfix=divb)
    edge = 16 if ndim == 2 else 8
    forest = AMRForest(ndim, (2 * edge,) * ndim, (edge,) * ndim, (0.0,) * ndim, (1.0,) * ndim, ("cont",) * (2 * ndim),
                       max_level=1)
    be = DeviceFV(par, forest)
    be.set_state(0, _low_pressure(par, be.shape))
    be.getbc(0)
    dt, ch = be.getdt_courant(0, 0.4)
    be.crash(clear=True)
    be.advect1(FS["hll"], 1.0, dt, ch, 0, 1, ("copy", 0))
    be.errest_flags(forest, AMRPar(refine_max_level=1, w_refine_weight={0: 1.0}))
    assert be.may_flag_small == may
    assert be.crash() == may
    be.close()
