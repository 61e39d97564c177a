"""Long walks of mesh instances are handed on: scenes whose points lie deep inside one instance or
inside several overlapping ones give the oracle's values, from one such packet to more of them than
there is room for."""
import numpy as np
import pytest

from ebgeometry_amd import BVHUnionIF, SphereSDF, Translate, TriMeshSDF
from ebgeometry_amd import workloads as wl
from oracle import port

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,deep", [(1, 1), (64, 64), (65, 1), (3000, 300), (150_000, 150_000)])
@pytest.mark.parametrize("instances", [1, 3])
def test_handed_on_instances(cuda, n, deep, instances):
    """Points about the common centre of 1 or 3 instances of a sphere-like mesh, where thousands of
    triangles are about as near; a small sphere there decides some values, and their sign."""
    import torch
    v, f = wl.displaced_icosphere(5, 15)
    m = TriMeshSDF(v, f)
    shifts = [np.array([0.01 * k, 0.02 * k, 0.0]) for k in range(instances)]
    u = BVHUnionIF([Translate(m, t) for t in shifts] + [SphereSDF([3.0, 0.0, 0.0], 0.5)])
    q = wl.mixed_queries(n, v, f, 16)
    q[:deep] *= 1e-3
    if n > 64:
        q[-32:] = (wl.near_surface(32, v, f, 1e-6, 17) + shifts[-1]).astype(np.float32)
    got = u.value(torch.from_numpy(q).to(cuda)).cpu().numpy().astype(np.float64)
    sub = np.unique(np.concatenate([np.linspace(0, n - 1, min(n, 600)), np.arange(max(0, n - 32), n)]).astype(np.int64))
    p = q[sub].astype(np.float64)
    o = port.Mesh(v.astype(np.float64), f)
    ref = np.minimum.reduce([o.sdf(p - t)[0] for t in shifts] + [np.linalg.norm(p - [3.0, 0.0, 0.0], axis=1) - 0.5])
    diag = float(np.linalg.norm(v.max(0).astype(np.float64) - v.min(0)))
    assert np.abs(got[sub] - ref).max() <= 1e-6 * diag
    sure = np.abs(ref) > 1e-6 * diag  # the shifted points are FP32
    assert np.array_equal(np.sign(got[sub][sure]), np.sign(ref[sure]))
