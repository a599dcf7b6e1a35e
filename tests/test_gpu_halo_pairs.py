"""The 3-D FP64 stage's halo pairs, loaded 16 bytes at a time where the stage
input allows it: an input aligned to 8 bytes only gives the same bits, over
periodic, copied, mirrored and sign-changing boundaries."""
from __future__ import annotations

import pytest
import torch

from amrvac_amd import problems
from amrvac_amd.host import FS, Par
from amrvac_amd.mesh import UniformMesh

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["fp64", "fp64_exact"])
@pytest.mark.parametrize("bz,limiter,flux", [(4, "cada3", "hll"), (10, "vanleer", "tvdlf"), (16, "koren", "hll")])
def test_stage_input_aligned_to_8_bytes(bz, limiter, flux, precision):
    from amrvac_amd.fv import DeviceFV
    print(f"[pairs] {bz} {limiter} {flux} {precision}", flush=True)
    par = Par(physics="mhd", ndim=3, ndir=3, gamma=5.0 / 3.0, typedivbfix="glm", flux_scheme=flux, limiter=limiter,
              typeboundspeed="Einfeldt", time_stepper="threestep", courantpar=0.5)
    mesh = UniformMesh(3, (32, 32, 2 * bz), (16, 16, bz), (0.0,) * 3, (1.0, 1.0, bz / 16.0),
                       ("periodic", "periodic", "symm", "cont", "asymm", "cont"), nghost=par.nghost)
    be = DeviceFV(par, mesh, precision=precision)
    w = torch.from_numpy(mesh.interior(problems.orszag_tang_3d(mesh)).copy()).cuda()
    pad = torch.empty(w.numel() + 1, dtype=torch.float64, device="cuda")
    odd = pad[1:].view(w.shape)
    odd.copy_(w)
    assert w.data_ptr() % 16 == 0 and odd.data_ptr() % 16 == 8
    torch.cuda.synchronize()
    dt, ch = be.getdt_state(w.data_ptr(), par.courantpar)
    out = []
    for u in (w, odd):
        o = torch.zeros_like(w)
        torch.cuda.synchronize()
        be.stage(FS[flux], 1.0, dt, ch, u.data_ptr(), o.data_ptr())
        be.sync()
        out.append(o)
    # the sign-changing boundary negates the density of its ghost cells too:
    # the faces next to it are NaN, in both
    assert torch.isfinite(out[0][4:]).all() and not torch.equal(out[0], w)
    assert torch.equal(out[0].view(torch.int64), out[1].view(torch.int64))
