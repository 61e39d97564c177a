"""Calls of few queries run narrow packets (1 to 32 queries per wavefront, unsorted at 1), and any
call may hand long walks on: at the sizes where the width changes, results are the oracle's."""
import numpy as np
import pytest

from ebgeometry_amd import TriMeshSDF
from ebgeometry_amd import workloads as wl
from oracle import port

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 4096, 4097, 8192, 8193, 16_385, 32_769, 65_537, 131_072, 131_073,
                               262_144, 262_145])
@pytest.mark.parametrize("faces", [False, True])
def test_every_packet_width(cuda, n, faces):
    import torch
    v, f = wl.displaced_icosphere(4, 51)
    q = wl.mixed_queries(n, v, f, 52)
    q[: max(1, n // 64)] *= 1e-3  # near the medial axis: long walks
    m = TriMeshSDF(v, f, leaf_size=8)
    r = m.query(torch.from_numpy(q).to(cuda), with_triangle=faces)
    d = (r[0] if faces else r).cpu().numpy().astype(np.float64)
    sub = np.unique(np.linspace(0, n - 1, min(n, 3000)).astype(np.int64))
    ref, tri = port.Mesh(v.astype(np.float64), f).sdf(q[sub].astype(np.float64))
    diag = float(np.linalg.norm(v.max(0).astype(np.float64) - v.min(0)))
    assert np.abs(d[sub] - ref).max() <= 1e-6 * diag
    assert np.array_equal(np.sign(d[sub][ref != 0]), np.sign(ref[ref != 0]))
    if faces:
        t = r[1].cpu().numpy()
        assert t.min() >= 0 and t.max() < f.shape[0]
