"""Taylor passes whose row arrays exceed what the caches hold (non-temporal loads of the
accumulator and the earlier powers): bit-identical to the tiled gather, above the line (81 MB
an array) and just below it."""
import numpy as np
import pytest

from helpers import random_packed, small_sphere
from octhip import api

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("order", [2, 4, 5])
@pytest.mark.parametrize("radius,lanes", [(4.0, 1024), (3.6, 1024)])
def test_taylor_matches_gather(gpu, radius, lanes, order):
    print(f"[taylor large rows radius={radius} order={order}]", flush=True)
    s = small_sphere(radius=radius, spacing=0.3, natoms=2, rc=1.2)
    assert (s.np * lanes * 8 > 64e6) == (radius == 4.0)
    f = random_packed(s.np_part, lanes, seed=order, np_inner=s.np)
    out = []
    for kernel in (2, 1):
        hm = api.HamiltonianDevice.from_system(s)
        hm.tune(kernel=kernel)
        psi = api.Batch(lanes // 2, s.np_part, True, lanes // 2, ff=gpu.from_numpy(f.copy()).cuda())
        api.Exponential(order).apply_batch(hm, psi, 0.01)
        out.append(psi.ff[: s.np].cpu().numpy())
    assert np.array_equal(out[0], out[1])
