"""The fused training step (tiles of 64 rows, partial gradients per workgroup, ordered sums) at the
edges of its tiles, and its reproducibility."""
import numpy as np
import pytest

from ebgeometry_amd import TriMeshSDF
from ebgeometry_amd import workloads as wl
from ebgeometry_amd._lib import check, lib
from oracle import mlp_ref, port
from test_gpu_mlp import norm_box, small_theta

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("samples", [1, 63, 64, 65, 127, 8191, 8192, 8193])
def test_gradient_at_tile_edges(cuda, samples):
    """One row, whole and ragged tiles, one tile per workgroup (8192 rows) and one more. The bar is
    the one of the larger gradients against the oracle, whose rounding points are the kernel's."""
    import torch
    v, f = wl.displaced_icosphere(3, 3)
    m = TriMeshSDF(v, f)
    theta = small_theta(2)
    m.set_bound_params(theta)
    q = wl.mixed_queries(samples, v, f, 6)
    d_ref, _ = port.Mesh(v.astype(np.float64), f).sdf(q.astype(np.float64))
    target = np.abs(d_ref).astype(np.float32)
    qt, tt = torch.from_numpy(q).to(cuda), torch.from_numpy(target).to(cuda)
    grads = []
    for _ in range(2):
        g = torch.zeros(int(lib().ebg_mlp_param_count()), dtype=torch.float32, device=cuda)
        loss = torch.zeros(1, dtype=torch.float32, device=cuda)
        check(lib().ebg_mlp_loss_grad(m.handle, qt.data_ptr(), tt.data_ptr(), samples, g.data_ptr(),
                                      loss.data_ptr(), None))
        torch.cuda.synchronize()
        grads.append(g.cpu().numpy())
    assert np.array_equal(grads[0], grads[1])  # sums in a fixed order
    lo, sc, diag = norm_box(m)
    L, gref = mlp_ref.loss_and_grad(theta.astype(np.float64), q, target, lo, sc, float(diag), bf16_mode=True)
    # a row whose BF16 rounding falls the other way moves its own share of the sums: with one row
    # that share is all of it (a BF16 step is 2^-8, and an activation passes four layers)
    rel = 2e-2 if samples > 1000 else 8e-2
    assert loss.item() / samples == pytest.approx(L, rel=max(2e-3, rel / 4))
    o = 0
    for shape in mlp_ref.SHAPES:
        k = int(np.prod(shape))
        a, b = grads[0][o:o + k].astype(np.float64), gref[o:o + k]
        assert np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-12) < rel, (shape, o)
        o += k


def test_training_is_reproducible(cuda):
    v, f = wl.displaced_icosphere(3, 9)
    w = []
    for _ in range(2):
        m = TriMeshSDF(v, f)
        m.train_bound(num_samples=5000, epochs=2, batch=1000, seed=4)
        w.append(m.get_bound_params())
    assert np.isfinite(w[0]).all() and np.array_equal(w[0], w[1])


def test_weights_are_written_when_training_returns(cuda):
    """A stream that does not wait for the training's (a torch stream: non-blocking) predicts with the
    trained weights at once."""
    import torch
    v, f = wl.displaced_icosphere(3, 9)
    q = torch.from_numpy(wl.mixed_queries(5000, v, f, 10)).to(cuda)
    side = torch.cuda.Stream()
    m = TriMeshSDF(v, f)
    for seed in range(8):
        m.train_bound(num_samples=4096, epochs=1, batch=4096, seed=seed)
        with torch.cuda.stream(side):
            at_once = m.predict_bound(q)
        torch.cuda.synchronize()
        assert torch.equal(at_once, m.predict_bound(q)), seed


def test_small_trainings_measure_no_cost_grid(cuda):
    """The first training of a mesh takes about as long as the second (0.9 ms; a cost grid, measured
    once, adds 5 ms on these faces)."""
    import time

    v, f = wl.displaced_icosphere(6, 3)
    first, again = [], []
    for k in range(6):
        m = TriMeshSDF(v, f)
        for t in (first, again):
            t0 = time.perf_counter()
            m.train_bound(num_samples=8192, epochs=1, batch=4096)
            t.append(time.perf_counter() - t0)
    assert np.median(first[1:]) < 2 * np.median(again[1:]) + 1e-3
