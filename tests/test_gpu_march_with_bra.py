"""The H-apply whose z-march takes the bra along and whose ket adds to the output rows:
bit-identical to the general path (tiled gather, bra and ket in launches of their own in front
of it) over the sphere layouts of the bra's group and block edges, the last of an odd number of
bra blocks, sets whose sums are too many to go along, and boundary rows cleared or taken as
they are."""
import numpy as np
import pytest

from helpers import random_packed
from octhip import api, periodic as PER
from test_gpu_ket_sets import LAYOUTS, system
from test_gpu_periodic import make

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("set_bc", [False, True])
@pytest.mark.parametrize("lanes", [8, 16, 32, 64])
@pytest.mark.parametrize("name", list(LAYOUTS))
def test_apply_matches_general_path(gpu, name, lanes, set_bc):
    print(f"[march with bra {name} lanes={lanes} set_bc={set_bc}]", flush=True)
    s = system(name)
    f = random_packed(s.np_part, lanes, seed=lanes)
    out = []
    for kernel in (2, 1):
        hm = api.HamiltonianDevice.from_system(s)
        hm.tune(kernel=kernel)
        psi = api.Batch(lanes // 2, s.np_part, True, lanes // 2, ff=gpu.from_numpy(f.copy()).cuda())
        h = api.Batch(lanes // 2, s.np, True, lanes // 2)
        api.hamiltonian_elec_apply_batch(hm, psi, h, set_bc=set_bc)
        out.append((h.ff.cpu().numpy(), psi.ff.cpu().numpy()))
    assert np.array_equal(out[0][0], out[1][0])
    assert np.array_equal(out[0][1], out[1][1])
    assert np.array_equal(out[0][1][: s.np], f[: s.np])
    assert np.array_equal(out[0][1][s.np:], 0.0 * f[s.np:] if set_bc else f[s.np:])


@pytest.mark.parametrize("nst", [4, 8, 16, 32])
def test_bloch_phases_match_general_path(gpu, nst):
    """A state without its Bloch phase (the march leaves the ket's rows for the ket to multiply)
    and a propagation step on one that carries it (no phase at the end)."""
    print(f"[march with bra, Bloch phases nst={nst}]", flush=True)
    s = PER.periodic_system(n=19, spacing=0.35, natoms=3, nwells=2, rc=1.3, seed=77)
    f = random_packed(s.np_part, 2 * nst, seed=nst)
    out = []
    for kernel in (2, 1):
        hm = make(s, k=np.array([-0.4, 0.15, 0.3]))
        hm.tune(kernel=kernel)
        psi, step = (api.Batch(nst, s.np_part, True, nst, ff=gpu.from_numpy(f.copy()).cuda()) for _ in range(2))
        h = api.Batch(nst, s.np, True, nst)
        api.hamiltonian_elec_apply_batch(hm, psi, h)
        api.Exponential(3).apply_batch(hm, step, 0.01)
        out.append([b.ff[: s.np].cpu().numpy() for b in (h, step)])
    assert np.array_equal(out[0][0], out[1][0])
    assert np.array_equal(out[0][1], out[1][1])
