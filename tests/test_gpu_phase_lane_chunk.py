"""A k-point apply at every lane chunk that tuning accepts.

A chunk of one lane holds no (re, im) pair, so its z-march cannot multiply a row by the Bloch
phase and a pass over the result does.  Bar: max relative error <= 1e-12 per state against the
oracle, with projectors.
"""
import numpy as np
import pytest

import oracle as O
from helpers import max_rel_err
from octhip import api, periodic as PER, workloads
from test_gpu_periodic import make

pytestmark = pytest.mark.gpu

K = np.array([0.2, 0.35, -0.1])


@pytest.fixture(scope="module")
def cell():
    return PER.periodic_system(n=18, spacing=0.35, natoms=2, nwells=2, rc=1.2, seed=41)


@pytest.mark.parametrize("lane_chunk", [1, 2, 4, 32])
@pytest.mark.parametrize("nst", [1, 5, 16])
def test_phased_apply_by_lane_chunk(gpu, cell, nst, lane_chunk):
    print(f"[phased apply nst={nst} lane_chunk={lane_chunk}]", flush=True)
    s = cell
    hm = make(s, k=K)
    hm.tune(lane_chunk=lane_chunk)
    rng = np.random.default_rng(nst)
    z = rng.standard_normal((nst, s.np)) + 1j * rng.standard_normal((nst, s.np))
    psib = api.Batch.from_states(z, s.np_part)
    hpsib = api.Batch(nst, s.np, True)
    api.hamiltonian_elec_apply_batch(hm, psib, hpsib)
    gpu.cuda.synchronize()
    phase, corr = s.phases(K)
    ref = O.periodic_apply(O.Hamiltonian(s.op, s.v, None), workloads.pack(z, s.np_part), s.bnd_src, s.proj, phase,
                           corr, s.pphase_of(K), has_phase=False)
    assert max_rel_err(hpsib.ff.cpu().numpy(), ref) <= 1e-12
