"""The z-march pass at the edges of its tiles and segments: bit-identical to the tiled gather
kernel (the general path, same bra and ket kernels) for every segment length around its
pipeline depths (a segment of one plane, shorter than the four partial sums, one more than the
unrolled loop), lane chunks with and without the lane-quad broadcasts, rows read as the caller
set them, and every epilogue."""
import numpy as np
import pytest

from helpers import random_packed, small_sphere
from octhip import api

pytestmark = pytest.mark.gpu


def handles(s, **knobs):
    zm, ga = api.HamiltonianDevice.from_system(s), api.HamiltonianDevice.from_system(s)
    zm.tune(kernel=2, **knobs)
    ga.tune(kernel=1)
    return zm, ga


def batch(gpu, host, nst):
    return api.Batch(nst, host.shape[0], True, host.shape[1] // 2, ff=gpu.from_numpy(host.copy()).cuda())


@pytest.mark.parametrize("zseg", [1, 2, 3, 4, 5, 8, 9, 13])
@pytest.mark.parametrize("lanes,knobs", [(2, {}), (8, {}), (16, {}), (16, dict(lanes_per_thread=1)),
                                         (64, dict(lane_chunk=32)), (64, dict(lane_chunk=4))])
def test_apply_matches_gather(gpu, zseg, lanes, knobs):
    print(f"[zmarch apply zseg={zseg} lanes={lanes} {knobs}]", flush=True)
    s = small_sphere(radius=3.1, spacing=0.31, natoms=3, rc=1.3)
    zm, ga = handles(s, zseg=zseg, **knobs)
    f = random_packed(s.np_part, lanes, seed=zseg)
    for set_bc in (False, True):
        out = []
        for hm in (zm, ga):
            psi, h = batch(gpu, f, lanes // 2), api.Batch(lanes // 2, s.np, True, lanes // 2)
            api.hamiltonian_elec_apply_batch(hm, psi, h, set_bc=set_bc)
            out.append(h.ff.cpu().numpy())
        assert np.array_equal(out[0], out[1])


@pytest.mark.parametrize("zseg", [1, 4, 9])
@pytest.mark.parametrize("order", [1, 2, 3, 4, 6])
@pytest.mark.parametrize("lanes,knobs", [(2, {}), (16, dict(lanes_per_thread=1)), (32, {})])
def test_taylor_matches_gather(gpu, zseg, order, lanes, knobs):
    print(f"[zmarch taylor zseg={zseg} order={order} lanes={lanes} {knobs}]", flush=True)
    s = small_sphere(radius=2.6, spacing=0.3, natoms=2, rc=1.2)
    f = random_packed(s.np_part, lanes, seed=order, np_inner=s.np)
    w = np.linspace(0.5, 1.5, lanes // 2)
    out = []
    for hm in handles(s, zseg=zseg, **knobs):
        te = api.Exponential(order)
        plain, first, second = (batch(gpu, f, lanes // 2) for _ in range(3))
        te.apply_batch(hm, plain, 0.01)
        rho = gpu.zeros(s.np, dtype=gpu.float64, device="cuda")
        te.apply_batch(hm, first, 0.01, psib2=second, deltat2=0.02, density=rho, weights=w)
        out.append([b.ff[: s.np].cpu().numpy() for b in (plain, first, second)] + [rho.cpu().numpy()])
    for a, b in zip(out[0][:3], out[1][:3]):
        assert np.array_equal(a, b)
    # the density's partial sums differ in order: lanes // 2 positive terms
    assert np.max(np.abs(out[0][3] - out[1][3])) <= lanes * 2.3e-16 * np.max(out[1][3])
