"""Work buffers whose growth to longer rows fails: shorter rows, which worked before, work after.

Each allocation of the growth fails in turn; the call returns its error and the next one, at
the length that the handle had buffers for, gives the oracle's result (<= 1e-12 per state).
"""
import pytest

import oracle as O
from helpers import max_rel_err, small_sphere
from octhip import _lib, api, workloads

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("what", ["apply", "taylor"])
def test_shorter_rows_work_after_a_failed_growth(gpu, what):
    s = small_sphere(radius=3.0, spacing=0.3, natoms=3, rc=1.2)
    z = workloads.gaussian_envelope_states(s, 32, width=2.0)
    oh = O.Hamiltonian(s.op, s.v, s.proj)
    ref = workloads.pack(z[:8], s.np_part)
    ref = oh.apply(ref) if what == "apply" else (oh.taylor(ref, 0.01, 4), ref[: s.np])[1]

    def run(hm, n):
        b = api.Batch.from_states(z[:n], s.np_part)
        if what == "taylor":
            api.Exponential(4).apply_batch(hm, b, 0.01)
            return b.ff[: s.np]
        out = api.Batch(n, s.np, True)
        api.hamiltonian_elec_apply_batch(hm, b, out)
        return out.ff

    failed = 0
    for k in range(20):
        print(f"[failed growth {what} allocation {k}]", flush=True)
        hm = api.HamiltonianDevice.from_system(s)
        run(hm, 8)
        if what == "taylor":  # the projector buffers are there: the Taylor powers' growth fails
            b = api.Batch.from_states(z, s.np_part)
            api.hamiltonian_elec_apply_batch(hm, b, api.Batch(32, s.np, True))
        _lib.call("octhip_inject_alloc_failure", k)
        try:
            run(hm, 32)
            done = True
        except _lib.OcthipError as e:
            assert e.code == _lib.ERR_ALLOC
            done = False
        finally:
            _lib.call("octhip_inject_alloc_failure", -1)
        got = run(hm, 8)
        gpu.cuda.synchronize()
        assert max_rel_err(got.cpu().numpy(), ref) <= 1e-12
        if done:
            break
        failed += 1
    assert done and failed >= 3
