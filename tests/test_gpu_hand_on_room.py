"""More long walks than there is room to hand on, over deep trees: the wavefronts that find no room
walk on within their stacks (no status word is set), and all values are the oracle's."""
import ctypes as C

import numpy as np
import pytest

from ebgeometry_amd import BVHUnionIF, MeshBatch, SphereSDF, Translate, TriMeshSDF
from ebgeometry_amd import workloads as wl
from ebgeometry_amd._lib import check, lib
from oracle import port

pytestmark = pytest.mark.gpu

N = 100_000  # some 1,600 packets; the lists hold the stacks of about 700


@pytest.fixture(scope="module")
def sphere():
    """327,680 faces, points next to the centre, where every triangle is about as near."""
    v, f = wl.icosphere(7)
    q = (wl.mixed_queries(N, v, f, 7) * np.float32(1e-4)).astype(np.float32)
    sub = np.unique(np.linspace(0, N - 1, 100).astype(np.int64))
    ref, _ = port.Mesh(v.astype(np.float64), f).sdf(q[sub].astype(np.float64))
    # an FP32 distance is within 2^-21 (d + 2 h) of the triangle's (h: the longest edge, 0.01 here)
    return v, f, q, sub, ref, 2.0 ** -21 * (1.0 + 2 * 0.01)


@pytest.mark.parametrize("K,leaf", [(4, 1), (4, 2), (8, 1), (8, 4)])
@pytest.mark.parametrize("kind", ["mesh", "plan", "scene"])
def test_no_room_on_a_deep_tree(cuda, sphere, kind, K, leaf):
    import torch
    v, f, q, sub, ref, tol = sphere
    x = torch.from_numpy(q).to(cuda)
    if kind == "plan":
        b = MeshBatch([(v, f)], branching=K, leaf_size=leaf)
        h = C.c_void_p()
        check(lib().ebg_batch_mesh(b.handle, 0, C.byref(h)))
        d = b.plan([(0, x)], workgroup=256).launch()[0]
    else:
        m = TriMeshSDF(v, f, branching=K, leaf_size=leaf)
        h = m.handle
        if kind == "mesh":
            d = m.query(x)
        else:
            u = BVHUnionIF([Translate(m, [0.0, 0.0, 0.0]), SphereSDF([9.0, 0.0, 0.0], 0.5)])
            d = u.value(x)
    torch.cuda.synchronize()
    assert lib().ebg_mesh_check(h) == 0
    assert np.abs(d.cpu().numpy()[sub].astype(np.float64) - ref).max() <= tol
