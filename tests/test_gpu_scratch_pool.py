"""The pooled scratch of calls without a handle serves every row length: once a call has run,
the same call allocates nothing."""
import numpy as np
import pytest

from octhip import _lib, api

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("pack", [1, 16, 512])
def test_a_second_call_allocates_nothing(gpu, pack):
    print(f"[scratch pool pack={pack}]", flush=True)
    rows, nvec = 300, 5
    r = np.random.default_rng(pack)
    dev = lambda: api.Batch(pack, rows, True, pack,  # noqa: E731
                            ff=gpu.from_numpy(r.standard_normal((rows, 2 * pack))).cuda())
    xs, phi = [dev() for _ in range(nvec)], dev()
    again = phi.clone()
    ov, norm = api.mesh_batch_orthogonalization(0.1, xs, phi, rows, normalize=True)
    _lib.call("octhip_inject_alloc_failure", 0)
    try:
        ov2, norm2 = api.mesh_batch_orthogonalization(0.1, xs, again, rows, normalize=True)
    finally:
        _lib.call("octhip_inject_alloc_failure", -1)
    assert np.array_equal(ov, ov2) and np.array_equal(norm, norm2)
    assert gpu.equal(phi.ff, again.ff)
