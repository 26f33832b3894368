"""Projector routes that the other systems' sphere layouts do not take: the bra by spheres with
Bloch phases, and a batched launch over systems of both kinds.

So many spheres on one point that its set does not fit the sums of a bra workgroup make a
Hamiltonian's bra go by spheres.  Bars: max relative error <= 1e-12 per state against the
oracle; batched launches bit-identical to per-pair calls.
"""
import dataclasses

import numpy as np
import pytest

import oracle as O
from helpers import max_rel_err, synthetic_projectors
from octhip import api, periodic as PER, workloads
from test_gpu_periodic import make
from test_gpu_ket_sets import system

pytestmark = pytest.mark.gpu

K = np.array([0.25, -0.3, 0.15])


@pytest.fixture(scope="module")
def cell():
    s = PER.periodic_system(n=16, spacing=0.35, natoms=0, nwells=2, rc=1.2, seed=17)
    centers = [(0.05 * i, 0.0, -0.04 * i) for i in range(24)]
    proj = synthetic_projectors(s.mesh, centers, 1.2, [4, 3, 4, 1] * 6, 29)
    r = np.random.default_rng(31)
    pphase = np.exp(1j * r.uniform(-np.pi, np.pi, len(proj.maps)))
    return dataclasses.replace(s, proj=proj, pphase_of=lambda k: pphase)


@pytest.mark.parametrize("kernel", [0, 1])
@pytest.mark.parametrize("has_phase", [False, True])
@pytest.mark.parametrize("nst", [2, 8, 16, 24])
def test_bra_by_spheres_with_phases(gpu, cell, nst, has_phase, kernel):
    print(f"[bra by spheres, phases nst={nst} has_phase={has_phase} kernel={kernel}]", flush=True)
    s = cell
    hm = make(s, k=K, kernel=kernel)
    r = np.random.default_rng(nst)
    z = r.standard_normal((nst, s.np)) + 1j * r.standard_normal((nst, s.np))
    phase, corr = s.phases(K)
    psi = workloads.pack(z, s.np_part)
    psib = api.Batch.from_states(z, s.np_part)
    out = api.Batch(nst, s.np, True)
    api.hamiltonian_elec_apply_batch(hm, psib, out, has_phase=has_phase)
    gpu.cuda.synchronize()
    ref = O.periodic_apply(O.Hamiltonian(s.op, s.v, None), psi, s.bnd_src, s.proj, phase, corr, s.pphase_of(K),
                           has_phase=has_phase)
    assert max_rel_err(out.ff.cpu().numpy(), ref) <= 1e-12


@pytest.mark.parametrize("nsts", [(8, 16), (24, 8), (16, 16)])
def test_batched_systems_of_both_kinds(gpu, nsts):
    print(f"[batched, bra by spheres and by sets {nsts}]", flush=True)
    pairs = []
    for name, nst in zip(("dense", "chain"), nsts):
        s = system(name)
        z = workloads.gaussian_envelope_states(s, nst, width=2.0)
        pairs.append((api.HamiltonianDevice.from_system(s), api.Batch.from_states(z, s.np_part), s, z))
    bp = api.BatchedPropagator([(hm, b) for hm, b, _, _ in pairs], 1e-3)
    bp.apply()
    for (hm, b, s, z), hp in zip(pairs, bp.hpsi):
        ref = api.Batch(b.nst, s.np, True, b.pack_size)
        api.hamiltonian_elec_apply_batch(hm, b, ref)
        gpu.cuda.synchronize()
        assert gpu.equal(hp.ff, ref.ff)
        host = O.Hamiltonian(s.op, s.v, s.proj).apply(workloads.pack(z, s.np_part))
        assert max_rel_err(hp.ff.cpu().numpy(), host) <= 1e-12
    twin = [(hm, b.clone()) for hm, b, _, _ in pairs]
    bp.taylor_step()
    for (_, b, s, _), (hm, e) in zip(pairs, twin):
        api.Exponential(4).apply_batch(hm, e, 1e-3)
        gpu.cuda.synchronize()
        assert gpu.equal(b.ff[: s.np], e.ff[: s.np])
