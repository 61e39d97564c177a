"""Programs are given LDS for the stack depth they reach, and those without tree walks run a kernel
of their own: from one value to the deepest stack, with and without saved points."""
import numpy as np
import pytest

import ebgeometry_amd as E
from oracle import csg_ref

pytestmark = pytest.mark.gpu


def nested(depth, transform):
    """A chain whose evaluation holds `depth` values (and saved points) at once."""
    f = E.Complement(E.SphereSDF([0.3, 0.1, -0.2], 0.6))
    for k in range(depth):
        s = E.SphereSDF([0.1 * k - 0.4, 0.05 * k, 0.0], 0.3 + 0.02 * k)
        f = E.Difference(s, f) if k % 2 else E.SmoothUnion([s, f], 0.1)
        if transform:
            f = E.Translate(f, [0.01 * k, -0.02, 0.01])
    return f


@pytest.mark.parametrize("n", [1, 128, 129, 255, 257, 2000])
@pytest.mark.parametrize("depth,transform", [(0, False), (0, True), (1, False), (3, True), (7, True), (9, False)])
def test_stack_depths(cuda, n, depth, transform):
    f = nested(depth, transform)
    q = np.random.default_rng(depth).uniform(-2, 2, (n, 3)).astype(np.float32)
    ref = csg_ref.evaluate(f, q, {})
    span = float(np.linalg.norm([4.0] * 3))
    v = f.value(q)
    assert np.abs(v - ref).max() <= 1e-5 * span
    big = np.abs(ref) > 1e-6 * span
    assert np.array_equal(np.sign(v[big]), np.sign(ref[big]))
    assert np.abs(f.value(q, fp64_all=True) - ref).max() <= 1e-7 * span


def test_programs_without_walks_reserve_no_sort(cuda):
    """Nothing is sorted for them: 2M points take a list of 8 MB, and none of the presort's arrays
    (72 MB)."""
    import torch
    f = nested(3, True)
    f.value(torch.zeros(8, 3, device=cuda))  # the program's own arrays
    q = torch.rand(2_000_000, 3, device=cuda)
    out = torch.empty(2_000_000, device=cuda)
    torch.cuda.synchronize()
    before, _ = torch.cuda.mem_get_info()
    f.value(q, out=out)
    torch.cuda.synchronize()
    after, _ = torch.cuda.mem_get_info()
    assert before - after < 24 << 20
