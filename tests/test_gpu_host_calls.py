"""Host-array calls share one buffer of the handle: sizes up and down, several threads at once, and calls
after a refused one give the values of the device-array call; a large call's buffer is given back."""
import threading

import numpy as np
import pytest

from ebgeometry_amd import TriMeshSDF
from ebgeometry_amd import workloads as wl
from ebgeometry_amd._lib import EbgError

pytestmark = pytest.mark.gpu


def test_sizes_and_threads(cuda):
    import torch
    v, f = wl.displaced_icosphere(3, 33)
    m = TriMeshSDF(v, f)
    sets = [wl.mixed_queries(n, v, f, 34 + n) for n in (1, 5000, 64, 70_001, 3)]
    ref = [m.query(torch.from_numpy(q).to(cuda)).cpu().numpy() for q in sets]
    for q, r in zip(sets, ref):
        assert np.array_equal(m.signed_distance(q), r)
    bad = []

    def work(k):
        for rep in range(5):
            j = (k + rep) % len(sets)
            if not np.array_equal(m.signed_distance(sets[j]), ref[j]):
                bad.append((k, j))

    threads = [threading.Thread(target=work, args=(k,)) for k in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad


def test_large_buffers_are_given_back(cuda):
    """5M points take 80 MB of points and distances, above what the handle keeps (64 MiB). The query
    workspace, which it does keep, is grown by a device-array call first."""
    import torch
    v, f = wl.displaced_icosphere(2, 35)
    m = TriMeshSDF(v, f)
    q = wl.mixed_queries(5_000_000, v, f, 36)
    ref = m.query(torch.from_numpy(q).to(cuda)).cpu().numpy()
    torch.cuda.empty_cache()
    before, _ = torch.cuda.mem_get_info()
    got = m.signed_distance(q)
    after, _ = torch.cuda.mem_get_info()
    assert np.array_equal(got, ref)
    assert before - after < 32 << 20


def test_call_after_a_refused_one(cuda):
    """The learned bound of an untrained mesh is refused after the points were sent to the device; the
    next call, on another stream, has the buffer to itself."""
    import torch
    v, f = wl.displaced_icosphere(3, 37)
    m = TriMeshSDF(v, f)
    q = wl.mixed_queries(300_000, v, f, 38)
    ref = m.query(torch.from_numpy(q).to(cuda)).cpu().numpy()
    side = torch.cuda.Stream()
    for _ in range(3):
        with pytest.raises(EbgError):
            m.signed_distance(q[::-1].copy(), learned_bound=True)
        assert np.array_equal(m.signed_distance(q, stream=side.cuda_stream), ref)
