"""Mesh instances of a scene, and mesh leaves of a program, are walked over the mesh's cylinder
bounds by the whole wavefront: at the edges of packets and of leaves the values are the oracle's."""
import numpy as np
import pytest

from ebgeometry_amd import Complement, Offset, TriMeshSDF
from ebgeometry_amd import workloads as wl
from ebgeometry_amd.scene import instance_matrix
from oracle import port
from test_gpu_scene import check, gpu_scene, oracle_scene

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 63, 64, 65, 257])
@pytest.mark.parametrize("level,leaf", [(0, 1), (0, 16), (2, 5), (3, 16)])
def test_instances_at_packet_edges(cuda, n, level, leaf):
    """Meshes of 20 to 1280 faces, leaves of 1 to 16; points at every depth of the instances (their
    centres too, where all triangles are about as near) and next to their surfaces (FP64 pass)."""
    sc = wl.csg_scene(21 + level, n_spheres=3, n_boxes=2, n_meshes=3, mesh_level=level, extent=4.0)
    u, _ = gpu_scene(sc, leaf=leaf)
    _, _, diag = u.bounds()
    q = [wl.uniform_box(n, [0.0] * 3, [4.0] * 3, 31)]
    for i, (v, f) in enumerate(zip(sc.mesh_verts, sc.mesh_faces)):
        local = wl.near_surface(n, v, f, 1e-5, 41 + i).astype(np.float64)
        local[::3] *= np.linspace(0.0, 0.9, len(local[::3]))[:, None]
        q.append(sc.mesh_translate[i] + float(sc.mesh_scale[i]) * (local @ instance_matrix(sc.mesh_rot_deg[i])))
    o = oracle_scene(sc)
    for pts in q:
        pts = np.ascontiguousarray(pts, np.float32)
        check(u.value(pts), o.value(pts.astype(np.float64)), diag, f"n={n} level={level} leaf={leaf}")


@pytest.mark.parametrize("n", [1, 65, 3000])
def test_program_leaf_equals_mesh_query(cuda, n):
    """A mesh leaf of a program gives the mesh's own signed distance (complemented and offset)."""
    v, f = wl.displaced_icosphere(3, 61)
    m = TriMeshSDF(v, f)
    q = wl.mixed_queries(n, v, f, 62)
    q[: max(1, n // 50)] *= 1e-3
    ref, _ = port.Mesh(v.astype(np.float64), f).sdf(q.astype(np.float64))
    diag = float(np.linalg.norm(v.max(0).astype(np.float64) - v.min(0)))
    got = Complement(Offset(m, 0.01)).value(q).astype(np.float64)
    assert np.abs(got + (ref - 0.01)).max() <= 1e-6 * diag
