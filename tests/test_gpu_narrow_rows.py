"""Bra and ket products over rows of fewer than 16 lanes (a lane tile that is partly empty):
real and complex rows of 1 to 8 lanes against the oracle, over the sphere layouts of the group
and block edges.  Bar: max relative error <= 1e-12 per state, as for every H-apply.  Lanes past
the rows are not touched: the output lies between rows of a sentinel."""
import numpy as np
import pytest

import oracle as O
from helpers import max_rel_err
from octhip import api, workloads
from test_gpu_ket_sets import LAYOUTS, system

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nst,cplx", [(1, False), (2, False), (7, False), (1, True), (2, True), (4, True)])
@pytest.mark.parametrize("name", list(LAYOUTS))
def test_nonlocal_term(gpu, name, nst, cplx):
    print(f"[narrow rows {name} nst={nst} complex={cplx}]", flush=True)
    s = system(name)
    z = workloads.gaussian_envelope_states(s, nst, width=2.0)
    z = z if cplx else np.ascontiguousarray(z.real)
    hm = api.HamiltonianDevice.from_system(s)
    psib = api.Batch.from_states(z, s.np_part)
    L = psib.ff.shape[1]
    room = gpu.full((s.np + 32, L), 7.25, dtype=gpu.float64, device="cuda")
    hpsib = api.Batch(nst, s.np, cplx, psib.pack_size, ff=room[16:16 + s.np])
    api.hamiltonian_elec_apply_batch(hm, psib, hpsib, api.TERM_NON_LOCAL_POTENTIAL)
    gpu.cuda.synchronize()
    host = psib.ff.cpu().numpy()
    ref = O.Hamiltonian(s.op, s.v, s.proj).apply(host, O.TERM_NON_LOCAL)
    n = (2 if cplx else 1) * nst
    assert np.max(np.abs(ref)) > 0.0
    assert max_rel_err(hpsib.ff.cpu().numpy()[:, :n], ref[:, :n]) <= 1e-12
    room = room.cpu().numpy()
    assert np.all(room[:16] == 7.25) and np.all(room[16 + s.np:] == 7.25)
