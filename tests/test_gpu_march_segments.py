"""Segments at 32 lanes a chunk: 60 planes run and match the tiled gather bit for bit, 61 are
refused, and the message says which limit that is."""
import pytest

from helpers import small_sphere
from octhip import _lib, api, workloads

pytestmark = pytest.mark.gpu


def test_longest_segment_of_32_lanes(gpu):
    print("[segments at 32 lanes]", flush=True)
    s = small_sphere(radius=10.5, spacing=0.3, natoms=2)  # 71 planes: more than one segment
    hm = api.HamiltonianDevice.from_system(s)
    psib = api.Batch.from_states(workloads.gaussian_envelope_states(s, 16, width=2.0), s.np_part)
    out = {}
    for tune in (dict(kernel=1), dict(kernel=2, lane_chunk=32, zseg=60)):
        hm.tune(**tune)
        out[len(tune)] = api.Batch(16, s.np, True)
        api.hamiltonian_elec_apply_batch(hm, psib, out[len(tune)])
    gpu.cuda.synchronize()
    assert gpu.equal(out[1].ff, out[3].ff)
    hm.tune(zseg=61)
    with pytest.raises(_lib.OcthipError, match="at most 60 planes"):
        api.hamiltonian_elec_apply_batch(hm, psib, out[1])
