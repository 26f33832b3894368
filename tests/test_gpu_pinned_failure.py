"""A Lanczos step whose pinned host buffer cannot be allocated: the allocation goes through the
library's hook like every other one, the call returns its error, and the handle works after."""
import pytest

import oracle as O
from helpers import max_rel_err, small_sphere
from octhip import _lib, api, workloads

pytestmark = pytest.mark.gpu


def test_pinned_allocation_goes_through_the_hook(gpu):
    print("[pinned allocation failure]", flush=True)
    s = small_sphere(radius=3.0, spacing=0.3, natoms=3, rc=1.2)
    z = workloads.orthonormalise(workloads.gaussian_envelope_states(s, 8, width=2.0), s.mesh.vol_pp)
    te = api.Exponential(12, method="lanczos", lanczos_tol=1e-8)
    messages = []
    for k in range(50):
        hm = api.HamiltonianDevice.from_system(s)  # without buffers of an earlier attempt
        b = api.Batch.from_states(z, s.np_part)
        _lib.call("octhip_inject_alloc_failure", k)
        try:
            te.apply_batch(hm, b, 0.01)
            break
        except _lib.OcthipError as e:
            assert e.code == _lib.ERR_ALLOC
            messages.append(str(e))
        finally:
            _lib.call("octhip_inject_alloc_failure", -1)
        if "hipHostMalloc" in messages[-1]:
            te.apply_batch(hm, b, 0.01)
            break
    assert "hipHostMalloc" in messages[-1] and "injected" in messages[-1], messages
    gpu.cuda.synchronize()
    ref = workloads.pack(z, s.np_part)
    it, _ = O.lanczos_batch(O.Hamiltonian(s.op, s.v, s.proj), ref, 8, 0.01, 12, 1e-8, s.mesh.vol_pp)
    assert te.last_iterations == it
    assert max_rel_err(b.ff.cpu().numpy()[: s.np], ref[: s.np]) <= 1e-12
