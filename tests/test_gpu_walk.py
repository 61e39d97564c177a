"""The FP32 walk's cylinder bounds and triangle discs never cull the closest triangle: against the
oracle's FP64 distance of every query, the FP32 pass alone is within the FP32 evaluation error of
a distance, 2^-21 (|d| + 2 hmax) plus the rounding of d itself (hmax the longest edge), over mesh
shapes (curved, flat and axis-aligned, slivers, one leaf), trees (4- and 8-wide, leaves of 1 to
16), sizes from 1e-5 to 1e15 and positions away from the origin."""
import numpy as np
import pytest

from ebgeometry_amd import Build, TriMeshSDF
from ebgeometry_amd import workloads as wl
from oracle import port
from test_gpu_mesh import sliver_sphere

pytestmark = pytest.mark.gpu


def box_mesh(cells):
    """A cube of 12 cells^2 axis-aligned right triangles."""
    index, verts, faces = {}, [], []
    for axis in range(3):
        for side in (0, cells):
            for a in range(cells):
                for b in range(cells):
                    ids = []
                    for da, db in ((0, 0), (1, 0), (1, 1), (0, 1)):
                        p = [0, 0, 0]
                        p[axis], p[(axis + 1) % 3], p[(axis + 2) % 3] = side, a + da, b + db
                        p = tuple(p)
                        if p not in index:
                            index[p] = len(verts)
                            verts.append(p)
                        ids.append(index[p])
                    ids = ids if side else ids[::-1]
                    faces += [[ids[0], ids[1], ids[2]], [ids[0], ids[2], ids[3]]]
    return np.array(verts, np.float32) / np.float32(cells), np.array(faces, np.uint32)


def shapes(name):
    if name == "sphere":
        return wl.displaced_icosphere(4, 7)
    if name == "box":
        return box_mesh(9)
    if name == "slivers":
        return sliver_sphere(2, 1e-3)
    v = np.array([[0, 0, 0], [1, 0, 0], [0, 1, 0], [0, 0, 1]], np.float32)
    return v, np.array([[0, 2, 1], [0, 1, 3], [0, 3, 2], [1, 2, 3]], np.uint32)


@pytest.mark.parametrize("name,K,leaf,build", [("sphere", 4, 16, Build.SAH), ("sphere", 8, 5, Build.SAH),
                                               ("sphere", 4, 1, Build.Morton), ("sphere", 8, 8, Build.SAH_GPU),
                                               ("box", 4, 4, Build.SAH), ("box", 8, 16, Build.SAH),
                                               ("slivers", 4, 4, Build.SAH), ("tetrahedron", 4, 4, Build.SAH),
                                               ("tetrahedron", 8, 1, Build.SAH)])
@pytest.mark.parametrize("scale,offset", [(1.0, 0.0), (1.0, 300.0), (1e-5, 0.0), (1e-3, 0.0), (1e9, 0.0), (1e15, 0.0)])
def test_no_closest_triangle_is_culled(cuda, name, K, leaf, build, scale, offset):
    v, f = shapes(name)
    q = np.concatenate([wl.mixed_queries(1500, v, f, 5), 0.2 * wl.uniform_box(300, [-1] * 3, [1] * 3, 6),
                        wl.uniform_box(200, [-40] * 3, [40] * 3, 7)]).astype(np.float64)
    v = (v.astype(np.float64) * scale + offset).astype(np.float32)
    q = (q * scale + offset).astype(np.float32)
    m = TriMeshSDF(v, f, build=build, branching=K, leaf_size=leaf)
    d = m.query(q, fp64_recheck=False).astype(np.float64)
    ref, _ = port.Mesh(v.astype(np.float64), f).sdf(q.astype(np.float64))
    x = v.astype(np.float64)[f.astype(np.int64)]
    hmax = max(np.linalg.norm(x[:, (i + 1) % 3] - x[:, i], axis=1).max() for i in range(3))
    err = np.abs(np.abs(d) - np.abs(ref))
    tol = 2.0 ** -21 * (np.abs(ref) + 2 * hmax) + 2.0 ** -23 * np.abs(ref)
    bad = np.nonzero(err > tol)[0]
    assert bad.size == 0, (bad.size, q[bad[0]], d[bad[0]], ref[bad[0]])


def test_points_beyond_fp32_squares_and_nan(cuda):
    """Points whose squared distance overflows FP32, infinite and NaN points share wavefronts with
    ordinary ones: those keep their answers, the far ones come out infinite."""
    import torch
    v, f = wl.displaced_icosphere(4, 8)
    m = TriMeshSDF(v, f)
    q = wl.mixed_queries(1000, v, f, 9)
    plain = m.query(q)
    mixed = q.copy()
    mixed[::50, 0] = 1e25
    mixed[7::50, 1] = np.nan
    out = torch.zeros(q.shape[0], device=cuda)
    d = m.query(torch.from_numpy(mixed).to(cuda), out=out).cpu().numpy()
    keep = np.ones(q.shape[0], bool)
    keep[::50] = keep[7::50] = False
    assert np.abs(d[keep] - plain[keep]).max() <= 1e-6
    assert np.all(np.isinf(d[::50]))
