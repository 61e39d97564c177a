"""Every k of a nearest-neighbour query: the entries sit at the end of arrays of 1, 4, 8 or 16."""
import numpy as np
import pytest

from ebgeometry_amd import PointCloudBVH
from oracle import cloud_ref
from test_gpu_cloud import check_knn

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("k", list(range(1, 17)))
@pytest.mark.parametrize("branching", [4, 8])
@pytest.mark.parametrize("points,n,leaf", [(16, 1, 16), (17, 63, 1), (900, 65, 7), (5000, 500, 8)])
def test_every_k(cuda, k, points, n, leaf, branching):
    rng = np.random.default_rng(points + k)
    P = rng.normal(size=(points, 3)).astype(np.float32)
    P[1::5] = P[0::5][: len(P[1::5])]  # equal points: equal distances
    Q = np.concatenate([P[: n // 2], rng.normal(size=(n - n // 2, 3)).astype(np.float32)])
    c = PointCloudBVH(P, leaf_size=leaf, branching=branching)
    idx, d2 = c.knn(Q, k)
    _, rd = cloud_ref.knn(P, Q, k)
    check_knn(P, Q, idx, d2, rd, f"k={k}")
    assert all(len(set(r)) == k for r in idx.tolist())
    if k < points:
        si, sd = c.all_nearest_neighbors(k)
        sel = np.arange(0, points, max(1, points // 50))
        _, rs = cloud_ref.knn(P, P[sel], k, exclude=sel.tolist())
        check_knn(P, P[sel], si[sel], sd[sel], rs, f"self k={k}", exclude=sel)


def test_points_that_are_no_numbers(cuda):
    P = np.random.default_rng(1).normal(size=(300, 3)).astype(np.float32)
    Q = P[:130].copy()
    Q[::3, 1] = np.nan
    idx, d2 = PointCloudBVH(P).knn(Q, 3)
    ok = ~np.isnan(Q).any(1)
    assert np.array_equal(idx[ok][:, 0], np.arange(130)[ok])
    assert (idx[~ok] == 0xFFFFFFFF).all() and np.isinf(d2[~ok]).all()
