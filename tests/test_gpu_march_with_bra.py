"""The H-apply whose z-march takes the bra along and whose ket adds to the output rows:
bit-identical to the general path (tiled gather, bra and ket in launches of their own in front
of it) over the sphere layouts of the bra's group and block edges, the last of an odd number of
bra blocks, sets whose sums are too many to go along, and boundary rows cleared or taken as
they are."""
import numpy as np
import pytest

from helpers import random_packed
from octhip import api
from test_gpu_ket_sets import LAYOUTS, system

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
