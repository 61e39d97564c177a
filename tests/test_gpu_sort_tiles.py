"""The radix sort at the edges of its tile counts: the rows of counts are summed 1,024 tiles (of 4,096
keys) at a time."""
import numpy as np
import pytest

from ebgeometry_amd import morton_sort

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tiles", [1, 255, 256, 1024, 1025])
@pytest.mark.parametrize("rest", [-1, 0, 1])
@pytest.mark.parametrize("high", [3, 1 << 40])
def test_stable_order(cuda, tiles, rest, high):
    """One key less and one more than whole tiles, on either side of a whole chunk, with few and with
    many digits in use."""
    import torch
    n = 4096 * tiles + rest
    keys = np.random.default_rng(n).integers(0, high, n, dtype=np.int64)
    perm, sk = morton_sort(torch.from_numpy(keys).to(cuda))
    torch.cuda.synchronize()
    ref = np.argsort(keys, kind="stable")
    assert np.array_equal(perm.cpu().numpy().astype(np.int64), ref)
    assert np.array_equal(sk.cpu().numpy().view(np.int64), keys[ref])
