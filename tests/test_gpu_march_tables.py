"""Index tables of the z-march on a tall mesh, beyond 2^31 ints in the larger case."""
import numpy as np
import pytest

from octhip import api
from octhip.stencil import NLOperator, star_points

pytestmark = pytest.mark.gpu


def tall_mesh(tiles, height):
    """Two points, at the bottom and at the top, in each of tiles x tiles column tiles."""
    g = 8 * np.arange(tiles)
    inner = np.stack(np.meshgrid(g, g, [0, height - 1], indexing="ij"), axis=-1).reshape(-1, 3)
    pts = star_points(4)
    nb = inner[:, None, :] + pts[None, :, :]
    key = lambda c: ((c[..., 2].astype(np.int64) + 8) * 10000 + c[..., 1] + 8) * 10000 + c[..., 0] + 8  # noqa: E731
    ki = key(inner)
    kb = np.setdiff1d(np.unique(key(nb)), ki)
    bnd = np.stack([kb % 10000 - 8, kb // 10000 % 10000 - 8, kb // 10 ** 8 - 8], axis=1)
    coords = np.concatenate([inner, bnd]).astype(np.int32)
    order = np.argsort(key(coords))
    idx = order[np.searchsorted(key(coords)[order], key(nb))]
    n = len(inner)
    ri = (idx - np.arange(n)[:, None]).astype(np.int32)
    w = np.linspace(-1.0, 1.5, 25)
    op = NLOperator(n=25, w=w, nri=n, ri=ri, rimap=np.arange(n, dtype=np.int32),
                    rimap_inv=np.arange(n + 1, dtype=np.int32), np=n, np_part=len(coords), center=4)
    return op, coords, idx


@pytest.mark.parametrize("tiles,height", [(3, 20), (64, 2044)])
def test_tall_mesh(gpu, tiles, height):
    """The larger one has 4096 tiles of 2052 planes of 256 ints: above 2^31."""
    print(f"[tall mesh tiles={tiles} height={height}]", flush=True)
    op, coords, idx = tall_mesh(tiles, height)
    dev = api.NLOperatorDevice(op, star_points(4), coords)
    assert dev.uses_lattice
    f = np.random.default_rng(1).standard_normal((op.np_part, 2))
    fi = api.Batch(1, op.np_part, True, ff=gpu.from_numpy(f).cuda())
    got = {}
    for kernel in (2, 1):
        dev.tune(kernel=kernel)
        fo = api.Batch(1, op.np, True)
        api.nl_operator_operate_batch(dev, fi, fo, 1.0)
        gpu.cuda.synchronize()
        got[kernel] = fo.ff.cpu().numpy()
    assert np.array_equal(got[1], got[2])
    # 25 terms of a few units: rounding of the sums only
    assert np.max(np.abs(got[2] - np.einsum("j,pjl->pl", op.w, f[idx]))) <= 25 * 25 * 10.0 * 2.0 ** -53
