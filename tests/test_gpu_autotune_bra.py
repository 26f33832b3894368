"""The autotuner times the MFMA bra at every row length that it takes: on rows below 16 lanes
it goes by sets and is faster than the plain form, so tuning such a handle keeps it."""
import pytest

import oracle as O
from helpers import max_rel_err
from octhip import api, workloads

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nst", [1, 4])
def test_short_rows_keep_the_mfma_bra(gpu, tmp_path, nst):
    print(f"[autotune short rows nst={nst}]", flush=True)
    s = workloads.hamiltonian_system(radius=4.0, spacing=0.25, seed=5, nwells=4, natoms=12, rc=1.5)
    hm = api.HamiltonianDevice.from_system(s)
    z = workloads.gaussian_envelope_states(s, nst, width=2.0)
    psib = api.Batch.from_states(z, s.np_part)
    hm.autotune(psib.ldf, reps=20, force=True)
    api.tuning_save(tmp_path / "t.txt")
    line = [ln.split() for ln in (tmp_path / "t.txt").read_text().splitlines()
            if ln.split()[:4] == [str(s.np), str(s.np_part), "12", str(psib.ldf)]]
    assert line[0][9] == "1", line              # bra: 1 = MFMA, 0 = plain
    out = api.Batch(nst, s.np, True)
    api.hamiltonian_elec_apply_batch(hm, psib, out)
    gpu.cuda.synchronize()
    ref = O.Hamiltonian(s.op, s.v, s.proj).apply(workloads.pack(z, s.np_part))
    assert max_rel_err(out.ff.cpu().numpy(), ref) <= 1e-12
