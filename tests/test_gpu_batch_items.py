"""Long walks of a plan are handed on: plans with few and many of them give the oracle's values, on
every replay, whatever the launch."""
import numpy as np
import pytest

from ebgeometry_amd import MeshBatch
from ebgeometry_amd import workloads as wl
from oracle import port

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,deep", [(1, 1), (64, 64), (65, 1), (3000, 300), (60_000, 60_000)])
@pytest.mark.parametrize("opts", [{}, {"persistent": True}, {"with_triangle": True}, {"presort": False}])
def test_handed_on_walks(cuda, n, deep, opts):
    """`deep` points of each item lie next to the centre, where thousands of triangles are about as
    near: from one long walk to more than the plan has slots for."""
    import torch
    meshes, queries = [], []
    for k in range(2):
        v, f = wl.displaced_icosphere(4 + k, 80 + k)
        q = wl.mixed_queries(n, v, f, 90 + k)
        q[:deep] *= 1e-3
        meshes.append((v, f))
        queries.append(q)
    b = MeshBatch(meshes, branching=4, leaf_size=8)
    items = [(k, torch.from_numpy(q).to(cuda)) for k, q in enumerate(queries)]
    plan = b.plan(items, capture=True, **opts)
    for _ in range(3):
        outs = plan.launch()
        torch.cuda.synchronize()
        for k, (v, f) in enumerate(meshes):
            d = outs[k].cpu().numpy().astype(np.float64)
            sub = np.unique(np.linspace(0, n - 1, min(n, 800)).astype(np.int64))
            ref, _ = port.Mesh(v.astype(np.float64), f).sdf(queries[k][sub].astype(np.float64))
            diag = float(np.linalg.norm(v.max(0).astype(np.float64) - v.min(0)))
            assert np.abs(d[sub] - ref).max() <= 1e-6 * diag, k
            assert np.array_equal(np.sign(d[sub][ref != 0]), np.sign(ref[ref != 0])), k
