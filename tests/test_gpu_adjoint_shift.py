"""The adjoint stage of a cell does not depend on where in its block's tile the
cell lies: a periodic state moved by half a block along y gives the gradient
moved with it, bit for bit.  Compared are the rows 0..4 and 8..12 of every
block: their faces are all reversed in the first round of each dimension, so
that the order of every sum is the same at both places."""
from __future__ import annotations

import pytest
import torch

from amrvac_amd import adjoint
from amrvac_amd.fv import DeviceFV
from amrvac_amd.host import FS, Par
from amrvac_amd.mesh import UniformMesh

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("ndim,divb", [(2, "none"), (2, "glm"), (3, "none"), (3, "glm")])
def test_adjoint_stage_moves_with_the_state(ndim, divb, precision):
    print(f"[adjoint shift] {ndim}-D {divb} {precision}", flush=True)
    dims = (32,) * ndim
    mesh = UniformMesh(ndim, dims, (16,) * ndim, (0.0,) * ndim, (1.0,) * ndim, ("periodic",) * (2 * ndim))
    par = Par(physics="mhd", ndim=ndim, ndir=3, gamma=5.0 / 3.0, typedivbfix=divb, time_stepper="threestep",
              flux_scheme="hll", limiter="vanleer", courantpar=0.4)
    be = DeviceFV(par, mesh, precision=precision)
    g = torch.Generator(device="cuda").manual_seed(20261205)
    shape = (1,) + dims[::-1]

    def rand():
        return 2.0 * torch.rand(shape, generator=g, dtype=torch.float64, device="cuda") - 1.0
    rho, v, b = 1.0 + 0.2 * rand(), [0.3 * rand() for _ in range(3)], [0.5 * rand() for _ in range(3)]
    p = 1.0 + 0.2 * rand()
    e = p / (par.gamma - 1.0) + 0.5 * rho * sum(c * c for c in v) + 0.5 * sum(c * c for c in b)
    u = torch.cat([rho] + [rho * c for c in v] + [e] + b + ([0.1 * rand()] if divb == "glm" else []))
    lam = torch.cat([rand() for _ in range(par.nw)])
    idx = torch.as_tensor(adjoint.block_index(mesh), device="cuda")
    ydim = ndim - 1  # of [nw, (z,) y, x]

    def reverse(u, lam):
        ub, lb = (adjoint.to_blocks(w, idx).contiguous() for w in (u, lam))
        out = torch.empty_like(ub)
        torch.cuda.synchronize()
        be.adjoint1(FS["hll"], 1.0, 2.0e-3, ub.data_ptr(), lb.data_ptr(), 1.0, out.data_ptr(), ch=3.0)
        be.sync()
        return out
    here = reverse(u, lam)
    moved = reverse(torch.roll(u, 8, dims=ydim), torch.roll(lam, 8, dims=ydim))
    back = torch.roll(torch.arange(32, device="cuda"), 8)  # row of `here` that lies at each row of `moved`
    rows = torch.tensor([r for r in range(32) if r % 16 <= 4 or 8 <= r % 16 <= 12], device="cuda")
    f, m = (adjoint.from_blocks(w, idx, dims[::-1]) for w in (here, moved))
    assert torch.equal(m.index_select(ydim, rows), f.index_select(ydim, back[rows]))
