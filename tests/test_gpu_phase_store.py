"""H apply with Bloch phases on a batch without them: one pass sets the boundary rows and
the phased copy, and the z-march stores its rows times the conjugate phase.

Bars: boundary rows are the images exactly; max relative error <= 1e-12 per state against
the oracle (the H-apply bar), for every row width a z-march lane chunk has, both lanes per
thread and the tiled gather, and on a cell whose side does not divide into tiles.
"""
import numpy as np
import pytest

import oracle as O
from helpers import max_rel_err
from octhip import api, periodic as PER, workloads
from test_gpu_periodic import make

pytestmark = pytest.mark.gpu

K = np.array([-0.4, 0.15, 0.3])


@pytest.fixture(scope="module")
def cell():
    return PER.periodic_system(n=19, spacing=0.35, natoms=2, nwells=2, rc=1.2, seed=99)


@pytest.mark.parametrize("tune", [dict(), dict(lanes_per_thread=1), dict(kernel=1)])
@pytest.mark.parametrize("nst", [1, 2, 3, 8, 16, 40])
def test_phased_apply(gpu, cell, nst, tune):
    print(f"[phase store nst={nst} {tune}]", flush=True)
    s = cell
    hm = make(s, k=K)
    hm.tune(**tune)
    rng = np.random.default_rng(nst)
    z = rng.standard_normal((nst, s.np)) + 1j * rng.standard_normal((nst, s.np))
    psib = api.Batch.from_states(z, s.np_part)
    hpsib = api.Batch(nst, s.np, True)
    api.hamiltonian_elec_apply_batch(hm, psib, hpsib)
    gpu.cuda.synchronize()
    psi = psib.ff.cpu().numpy()
    assert np.array_equal(psi[s.np:], psi[s.bnd_src])
    phase, corr = s.phases(K)
    ref = O.periodic_apply(O.Hamiltonian(s.op, s.v, None), workloads.pack(z, s.np_part), s.bnd_src, s.proj, phase,
                           corr, s.pphase_of(K), has_phase=False)
    assert max_rel_err(hpsib.ff.cpu().numpy(), ref) <= 1e-12
