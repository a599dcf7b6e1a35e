"""How far a 3-D result depends on the workgroups: a block's planes are split
over several of them on a level of few blocks and left whole on one that fills
the GPU.  A periodic state on 2 blocks (a workgroup per plane) against the same
state repeated over 512 (whole blocks, two per compute unit), and the mixed
form's blocks, which stay whole, at two depths."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from amrvac_amd import adjoint
from amrvac_amd.fv import DeviceFV
from amrvac_amd.host import Par, TimeIntegrator
from amrvac_amd.mesh import UniformMesh

pytestmark = pytest.mark.gpu

CELLS = (32, 16, 16)  # the repeated level, 2 blocks


def _state(par, dims, seed=20261208):
    """Conserved fields [nwt, z, y, x] of a periodic flow with noise on every
    variable; with constrained transport the faces' field (divergence-free in
    the discrete sense: component d does not vary along d) after the cells."""
    rng = np.random.default_rng(seed)
    x, y, z = np.meshgrid(*[(np.arange(n) + 0.5) / n for n in dims], indexing="ij")
    x, y, z = (c.transpose(2, 1, 0) for c in (x, y, z))
    tp = 2.0 * np.pi

    def noise():
        return 1.0e-3 * rng.uniform(-1.0, 1.0, x.shape)
    rho, p = 1.0 + 0.2 * np.sin(tp * x) + noise(), 0.8 + 0.2 * np.cos(tp * (y + z)) + noise()
    v = [-np.sin(tp * y) + noise(), np.sin(tp * x) + noise(), 0.3 * np.sin(tp * (x + z)) + noise()]
    e = p / (par.gamma - 1.0) + 0.5 * rho * sum(c * c for c in v)
    w = [rho] + [rho * c for c in v]
    if par.physics == "hd":
        return np.stack(w + [e])
    b = [0.3 * np.sin(tp * y), 0.3 * np.sin(2.0 * tp * x), 0.2 * np.cos(tp * x)]
    if not par.stagger:
        b = [c + noise() for c in b]
    w += [e + 0.5 * sum(c * c for c in b)] + b
    if par.typedivbfix == "glm":
        w.append(0.1 * noise())
    return np.stack(w + (b if par.stagger else []))


def _advance(par, precision, u, block, steps):
    """u after `steps` steps on blocks of `block` cells, as fields."""
    dims = u.shape[:0:-1]
    mesh = UniformMesh(3, dims, block, (0.0,) * 3, tuple(n / 32.0 for n in dims), ("periodic",) * 6,
                       nghost=par.nghost)
    idx = torch.as_tensor(adjoint.block_index(mesh))
    w = np.zeros((mesh.nblocks, par.nwt) + mesh.nxg[::-1])
    mesh.interior(w)[...] = adjoint.to_blocks(torch.as_tensor(u), idx).numpy()
    be = DeviceFV(par, mesh, precision=precision)
    be.set_state(0, w)
    ti = TimeIntegrator(par, mesh, be)
    ti.run(nsteps=steps)
    out = torch.as_tensor(np.ascontiguousarray(mesh.interior(be.get_state(0))))
    be.close()
    return adjoint.from_blocks(out, idx, dims[::-1]).numpy(), ti.state.dts


def _split_and_whole(par, precision):
    u = _state(par, CELLS)
    split, dts = _advance(par, precision, u, (16, 16, 16), 1)
    rep = (8, 8, 4)  # along x, y, z: 512 blocks
    whole, dtw = _advance(par, precision, np.tile(u, (1,) + rep[::-1]), (16, 16, 16), 1)
    assert dts == dtw
    nx, ny, nz = CELLS
    return split, [whole[:, k * nz:(k + 1) * nz, j * ny:(j + 1) * ny, i * nx:(i + 1) * nx]
                   for k, j, i in ((0, 0, 0), (1, 3, 5), (3, 7, 7))]


def _par(physics, divb, flux, limiter, stepper="threestep", **kw):
    return Par(physics=physics, ndim=3, ndir=3, gamma=5.0 / 3.0, typedivbfix=divb, flux_scheme=flux, limiter=limiter,
               typeboundspeed="Einfeldt", time_stepper=stepper, courantpar=0.4, **kw)


@pytest.mark.parametrize("type_ct,flux,limiter", [
    ("average", "hll", "cada3"), ("uct_contact", "hll", "vanleer"), ("uct_contact", "tvdlf", "minmod"),
    ("uct_hll", "hlld", "cada3"), ("uct_hll", "tvdlf", "koren")])
@pytest.mark.parametrize("precision", ["mixed", "fp64_exact"])
def test_constrained_transport_split_equals_whole(type_ct, flux, limiter, precision):
    """Mixed: every FP32 face is rounded alike wherever it is formed."""
    print(f"[split] ct {type_ct} {flux} {limiter} {precision}", flush=True)
    split, parts = _split_and_whole(_par("mhd", "ct", flux, limiter, type_ct=type_ct), precision)
    for p in parts:
        assert np.array_equal(p, split)


@pytest.mark.parametrize("physics,divb,flux,limiter,stepper", [
    ("hd", "none", "hllc", "vanleer", "threestep"), ("mhd", "none", "hlld", "minmod", "threestep"),
    ("mhd", "glm", "hll", "vanleer", "threestep"), ("mhd", "glm", "hll", "weno5", "threestep"),
    ("mhd", "linde", "tvdlf", "minmod", "twostep")])
@pytest.mark.parametrize("precision", ["fp64", "fp64_exact"])
def test_fp64_split_equals_whole_to_rounding(physics, divb, flux, limiter, stepper, precision):
    """The production kernels may round a part's first z face apart from the
    same face inside a march: over the three stages of a step that is a few
    roundings of the two fluxes of a cell (limiters without a jump: cada3's two
    forms differ, and a last bit may decide between them)."""
    print(f"[split] {physics} {divb} {flux} {limiter} {precision}", flush=True)
    split, parts = _split_and_whole(_par(physics, divb, flux, limiter, stepper), precision)
    bound = 0.0 if precision == "fp64_exact" else 64.0 * 2.0 ** -53 * np.abs(split).max()
    for p in parts:
        assert np.abs(p - split).max() <= bound


@pytest.mark.parametrize("physics,divb,flux,limiter", [
    ("hd", "none", "tvdlf", "minmod"), ("hd", "none", "hllc", "weno5"), ("mhd", "none", "hll", "cada3"),
    ("mhd", "glm", "hll", "cada3"), ("mhd", "glm", "hll", "koren"), ("mhd", "none", "hllc", "vanleer"),
    ("mhd", "glm", "hlld", "vanleer"), ("mhd", "none", "hll", "weno5")])
def test_mixed_result_does_not_depend_on_the_blocks_depth(physics, divb, flux, limiter):
    """Both blocks at a shared z face form the same flux (all but ideal MHD with
    TVDLF, and with GLM and WENO5)."""
    print(f"[split] depth {physics} {divb} {flux} {limiter}", flush=True)
    par = _par(physics, divb, flux, limiter)
    u = _state(par, (32, 16, 32))
    (a, ta), (b, tb) = (_advance(par, "mixed", u, (16, 16, bz), 2) for bz in (16, 8))
    assert ta == tb
    assert np.array_equal(a, b)
