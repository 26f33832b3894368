"""Gram-Schmidt passes at their edges against numpy: numbers of vectors around the four a pass
takes (none, one, four, five, nine), row lengths from one state to more states than a workgroup
has threads, states that do not fill the row, fewer points than a workgroup has row groups, and
every choice of outputs.  Bars: overlaps and norms <= 1e-13 relative (sums of 10^3 products in
another order), states <= 1e-12."""
import ctypes as C

import numpy as np
import pytest

from octhip import _lib, api

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nvec", [0, 1, 4, 5, 9])
@pytest.mark.parametrize("pack,nst,rows", [(1, 1, 1000), (8, 5, 3), (16, 16, 1021), (512, 300, 97)])
def test_gram_schmidt(gpu, nvec, pack, nst, rows):
    print(f"[gram-schmidt nvec={nvec} pack={pack} nst={nst} rows={rows}]", flush=True)
    r = np.random.default_rng(nvec + pack)
    vol = 0.027
    x = [r.standard_normal((rows + 2, 2 * pack)) for _ in range(nvec)]
    y = r.standard_normal((rows + 2, 2 * pack))
    dev = lambda a: api.Batch(nst, rows + 2, True, pack, ff=gpu.from_numpy(a.copy()).cuda())  # noqa: E731
    z = lambda a: a[:rows].view(np.complex128)[:, :nst]  # noqa: E731
    ov = np.array([vol * np.sum(np.conj(z(a)) * z(y), axis=0) for a in x]).reshape(nvec, nst)
    ref = z(y) - sum((o[None, :] * z(a) for o, a in zip(ov, x)), np.zeros(nst))
    nrm = np.sqrt(vol * np.sum(np.abs(ref) ** 2, axis=0))
    for normalize in (False, True):
        xs, phi = [dev(a) for a in x], dev(y)
        got_ov, got_n = api.mesh_batch_orthogonalization(vol, xs, phi, rows, normalize=normalize)
        scale = max(1.0, float(np.max(np.abs(ov)))) if nvec else 1.0
        assert nvec == 0 or np.max(np.abs(got_ov - ov)) <= 1e-13 * scale
        assert np.max(np.abs(got_n - nrm)) <= 1e-12 * np.max(nrm)
        want = ref / nrm[None, :] if normalize else ref
        out = phi.ff.cpu().numpy()
        assert np.max(np.abs(z(out) - want)) <= 1e-12 * np.max(np.abs(want))
        # rows past the inner ones, and states past nst, are left alone
        assert np.array_equal(out[rows:], y[rows:])
        assert np.array_equal(out[:, 2 * nst:], y[:, 2 * nst:])
    # without outputs the states are the same
    phi2 = dev(y)
    ptrs = (C.c_void_p * max(nvec, 1))(*[b.ptr() for b in (dev(a) for a in x)]) if nvec == 0 else None
    if ptrs is None:
        keep = [dev(a) for a in x]
        ptrs = (C.c_void_p * nvec)(*[b.ptr() for b in keep])
    _lib.call("octhip_mesh_batch_orthogonalization", nvec, ptrs, phi2.ptr(), phi2.ldf, nst, rows, vol, 1, None, None,
              None)
    assert np.array_equal(phi2.ff.cpu().numpy(), out)
