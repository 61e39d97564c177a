"""The FP64 decision of closest faces and near-surface queries gathers its triangles over leaves
before it evaluates them: for leaves of every size, and for points with one and with very many
triangles about as near, distance and face are the oracle's."""
import numpy as np
import pytest

from ebgeometry_amd import TriMeshSDF
from ebgeometry_amd import workloads as wl
from oracle import port

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("leaf", [1, 2, 3, 7, 15, 16])
@pytest.mark.parametrize("level,n", [(0, 1), (0, 65), (2, 63), (4, 700)])
def test_closest_face(cuda, leaf, level, n):
    import torch
    v, f = wl.displaced_icosphere(level, 71)
    q = wl.mixed_queries(n, v, f, 72)
    q[::2] = wl.near_surface(len(q[::2]), v, f, 1e-6, 73)  # FP64 decides their sign
    q[::5] *= 1e-4                                         # and thousands of faces are within the band
    m = TriMeshSDF(v, f, leaf_size=leaf)
    d, t = m.closest_triangle(torch.from_numpy(q).to(cuda))
    d, t = d.cpu().numpy().astype(np.float64), t.cpu().numpy().astype(np.int64)
    o = port.Mesh(v.astype(np.float64), f)
    ref, _ = o.sdf(q.astype(np.float64))
    diag = float(np.linalg.norm(v.max(0).astype(np.float64) - v.min(0)))
    assert np.abs(d - ref).max() <= 1e-7 * diag
    assert np.array_equal(np.sign(d[ref != 0]), np.sign(ref[ref != 0]))
    assert t.min() >= 0 and t.max() < f.shape[0]
    # the face is one at the least distance (up to the rounding of an FP64 distance)
    for i in range(min(n, 60)):
        one, _ = port.Mesh(v.astype(np.float64), f[t[i]:t[i] + 1]).sdf(q[i:i + 1].astype(np.float64))
        assert abs(abs(one[0]) - abs(ref[i])) <= 1e-12 * diag
