"""Device memory of an adjoint: what include/octhip.h says, in batches of np rows."""
import gc

import numpy as np
import pytest

from helpers import small_sphere
from octhip import api

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nsteps,K,order", [(6, 2, 2), (5, 5, 1), (4, 1, 4)])
def test_adjoint_holds_what_it_says(gpu, nsteps, K, order):
    print(f"[adjoint memory nsteps={nsteps} K={K} order={order}]", flush=True)
    s = small_sphere(radius=5.0, spacing=0.25, natoms=1)
    hm = api.HamiltonianDevice.from_system(s)
    nst = 64
    ldf = int(np.log2(2 * nst))
    b = api.Batch(nst, s.np_part, True)
    hm.set_dipole_field([0.0, 0.0, 0.0], positions=s.mesh.x[: s.np])
    api.Exponential(4).apply_batch(hm, b, 0.01)  # the work buffers, which are the Hamiltonian's
    gc.collect()
    gpu.cuda.synchronize()
    gpu.cuda.empty_cache()
    free0 = gpu.cuda.mem_get_info()[0]
    adj = api.Adjoint(hm, s.mesh.x, [1.0, 0.0, 0.0], ldf, nsteps, 0.01, s.mesh.vol_pp, order=order, checkpoint_every=K)
    batches = -(-nsteps // K) + 2 * K + 2 * K * (order - 1) + 2 * order + 2
    rows = s.np * 2 * nst * 8
    used = free0 - gpu.cuda.mem_get_info()[0]
    # potentials, partial sums and the rounding of seven allocations: below half a batch
    assert abs(used - batches * rows) < rows / 2, f"{used / rows:.2f} batches held, {batches} stated"
    del adj
