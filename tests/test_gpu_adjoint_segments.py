"""The adjoint's last two segments, which the forward leaves for the backward.

The first backward after a forward takes them as they are, a second one recomputes every
segment from its checkpoint with the same kernels: both must agree bit for bit, for one,
two, three and more segments, a ragged last one and orders with and without kept terms.
A potential set in between is used for every segment, as the checkpoints' recomputation
does: the gradients are those of a backward that recomputes everything.
"""
import numpy as np
import pytest

from octhip import api
from test_gpu_adjoint import problem

pytestmark = pytest.mark.gpu


def gradients(gpu, adj, phib, psib, s, vol):
    from octhip.autograd import overlap_objective
    _, chib = overlap_objective(phib, psib, s.np, vol)
    deps, dv = adj.backward(chib)
    gpu.cuda.synchronize()
    return np.array(deps), dv.cpu().numpy(), chib.ff.cpu().numpy()


@pytest.mark.parametrize("K,nsteps,order", [(12, 12, 4), (6, 12, 4), (7, 12, 4), (4, 10, 4), (1, 5, 4), (2, 9, 1),
                                            (3, 7, 2), (3, 7, 6)])
def test_held_segments(gpu, K, nsteps, order):
    print(f"[adjoint segments K={K} nsteps={nsteps} order={order}]", flush=True)
    s, vol, psi0, phi, eps = problem(nsteps=nsteps)
    hm = api.HamiltonianDevice.from_system(s)
    adj = api.Adjoint(hm, s.mesh.x, [1.0, 0.0, 0.0], int(np.log2(psi0.shape[1])), nsteps, 0.01, vol, order=order,
                      checkpoint_every=K)
    psi0 = psi0.copy()
    psi0[s.np:] = 3.0                       # what the boundary rows hold does not matter ...
    psib = api.Batch(8, s.np_part, True, ff=gpu.from_numpy(psi0).cuda())
    phib = api.Batch(8, s.np_part, True, ff=gpu.from_numpy(phi.copy()).cuda())
    adj.forward(psib, eps)
    assert not psib.ff[s.np:].any()         # ... and they leave cleared
    held = gradients(gpu, adj, phib, psib, s, vol)
    again = gradients(gpu, adj, phib, psib, s, vol)
    for a, b in zip(held, again):
        assert np.array_equal(a, b)
    # a new potential between the two passes
    v2 = s.v * 1.25 + 0.1
    psib.ff.copy_(gpu.from_numpy(psi0))
    adj.forward(psib, eps)
    hm.set_potential(v2)
    held = gradients(gpu, adj, phib, psib, s, vol)
    again = gradients(gpu, adj, phib, psib, s, vol)
    for a, b in zip(held, again):
        assert np.array_equal(a, b)
