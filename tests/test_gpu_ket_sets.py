"""Bra and ket over mesh points grouped by the set of projector matrices they belong to.

Bar: max relative error <= 1e-12 per state against the oracle, as for every H-apply (the
sums are the oracle's in another grouping).  The sphere layouts take the group and block
edges: one sphere, a point set smaller than a group, disjoint spheres, sets of two and
three, sets of more than 16 projector rows with mixed counts, and so many spheres on
one point that its set no longer fits the sums of a bra workgroup.
"""
import dataclasses

import numpy as np
import pytest

import oracle as O
from helpers import max_rel_err, small_sphere, synthetic_projectors
from octhip import api, workloads

pytestmark = pytest.mark.gpu

LAYOUTS = {
    "one": ([(0.0, 0.0, 0.0)], 1.5, [4]),
    "tiny": ([(0.0, 0.0, 0.0), (1.2, 0.0, 0.0)], 0.2, [3, 5]),
    "disjoint": ([(-1.5, 0.0, 0.0), (1.5, 0.0, 0.0)], 0.9, [4, 4]),
    "chain": ([(-1.4, 0.0, 0.0), (-0.5, 0.0, 0.0), (0.5, 0.1, 0.0), (1.4, 0.0, 0.2)], 1.0, [4, 1, 6, 4]),
    "wide": ([(0.0, 0.0, 0.0), (0.4, 0.2, 0.0), (-0.3, 0.0, 0.5)], 1.3, [18, 7, 18]),
    "stack": ([(0.06 * i, 0.0, -0.05 * i) for i in range(12)], 1.2, [4, 2, 4, 1, 4, 4, 3, 4, 4, 4, 4, 4]),
    "dense": ([(0.05 * i, 0.0, -0.04 * i) for i in range(24)], 1.2, [4] * 24),
}


def system(name):
    centers, rc, counts = LAYOUTS[name]
    s = small_sphere(radius=3.0, spacing=0.3, natoms=0)
    return dataclasses.replace(s, proj=synthetic_projectors(s.mesh, centers, rc, counts, 5 + len(centers)))


@pytest.mark.parametrize("bra", [0, 1])
@pytest.mark.parametrize("nst", [1, 8, 16])
@pytest.mark.parametrize("name", list(LAYOUTS))
def test_nonlocal_term(gpu, name, nst, bra):
    print(f"[ket sets {name} nst={nst} bra={bra}]", flush=True)
    s = system(name)
    z = workloads.gaussian_envelope_states(s, nst, width=2.0)
    hm = api.HamiltonianDevice.from_system(s)
    hm.tune(bra_mode=bra)
    psib = api.Batch.from_states(z, s.np_part)
    hpsib = api.Batch(nst, s.np, True)
    api.hamiltonian_elec_apply_batch(hm, psib, hpsib, api.TERM_NON_LOCAL_POTENTIAL)
    gpu.cuda.synchronize()
    ref = O.Hamiltonian(s.op, s.v, s.proj).apply(workloads.pack(z, s.np_part), O.TERM_NON_LOCAL)
    assert np.max(np.abs(ref)) > 0.0
    assert max_rel_err(hpsib.ff.cpu().numpy(), ref) <= 1e-12


@pytest.mark.parametrize("bra", [0, 1])
@pytest.mark.parametrize("nst", [8, 16])
def test_infinity_stays_in_its_sphere(gpu, nst, bra):
    print(f"[ket sets infinity nst={nst} bra={bra}]", flush=True)
    s = system("chain")
    maps, off = np.asarray(s.proj.maps), np.asarray(s.proj.offsets).reshape(-1, 6)
    inside = [set(maps[o[3]: o[3] + o[0]] - 1) for o in off]
    bad = min(inside[0] - inside[1] - inside[2] - inside[3])   # a point of the first sphere only
    z = workloads.gaussian_envelope_states(s, nst, width=2.0)
    z[:, bad] = np.inf
    hm = api.HamiltonianDevice.from_system(s)
    hm.tune(bra_mode=bra)
    psib = api.Batch.from_states(z, s.np_part)
    hpsib = api.Batch(nst, s.np, True)
    api.hamiltonian_elec_apply_batch(hm, psib, hpsib, api.TERM_NON_LOCAL_POTENTIAL)
    gpu.cuda.synchronize()
    got = hpsib.ff.cpu().numpy()
    finite = np.isfinite(got).all(axis=1)
    first = np.zeros(s.np, dtype=bool)
    first[sorted(inside[0])] = True
    assert finite[~first].all()
    assert not finite[first].any()
