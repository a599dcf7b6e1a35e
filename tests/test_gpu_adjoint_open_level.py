"""The adjoint stage on a level whose neighbour table leaves out a neighbour,
although its boundaries are declared periodic: refused on the host."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from amrvac_amd.fv import DeviceFV, FVError
from amrvac_amd.host import FS, Par
from amrvac_amd.mesh import UniformMesh

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ndim,face", [(2, f) for f in range(4)] + [(3, f) for f in range(6)])
def test_adjoint_refuses_a_missing_neighbour(ndim, face):
    print(f"[adjoint open] {ndim}-D face {face}", flush=True)
    par = Par(physics="hd", ndim=ndim, ndir=ndim, gamma=1.4, time_stepper="threestep", flux_scheme="hll",
              limiter="vanleer")
    mesh = UniformMesh(ndim, (32,) * ndim, (16,) * ndim, (0.0,) * ndim, (1.0,) * ndim, ("periodic",) * (2 * ndim))
    # direction n = (i1 + 1) + 3 (i2 + 1) + 9 (i3 + 1)
    n = (3 ** ndim - 1) // 2 + (1 if face % 2 else -1) * 3 ** (face // 2)
    table = np.array(mesh.neighbor, copy=True).reshape(mesh.nblocks, -1)
    table[1, n] = -1
    mesh.neighbor = table.reshape(np.shape(mesh.neighbor))
    be = DeviceFV(par, mesh)
    u, lam, out = (torch.ones((mesh.nblocks, par.nw) + (16,) * ndim, dtype=torch.float64, device="cuda")
                   for _ in range(3))
    torch.cuda.synchronize()
    with pytest.raises(FVError, match="all neighbours"):
        be.adjoint1(FS["hll"], 1.0, 1.0e-3, u.data_ptr(), lam.data_ptr(), 1.0, out.data_ptr())
    be.close()
