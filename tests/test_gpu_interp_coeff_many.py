"""GPU: conservative quadratic interpolation at a negative monotonic coefficient in calls of many boxes, against the oracle."""
import numpy as np
import pytest

import oracle

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("size", [(12, 11, 10), (16, 16, 8), (8, 8, 2), (4, 4, 4)])
def test_negative_coefficient_of_many_boxes(size, dtype):
    """The same bits as of few boxes: the same operations in the same order."""
    from gamer_amd import hydro
    print(f"[gpu] cquad coefficient -1.5, 600 boxes of {size} {dtype.__name__}", flush=True)
    few, many = 5, 600
    cd = np.random.default_rng(42).standard_normal((few, 5) + tuple(n + 2 for n in reversed(size))).astype(dtype)
    fd = np.zeros((few, 5) + tuple(2 * n for n in reversed(size)), dtype=dtype)
    kw = dict(scheme="CQUAD", mono_coeff=-1.5, int_prim=False, reduce_mono=False)
    _, want, _ = oracle.interpolate(cd, fd, (1, 1, 1), size, **kw)
    at = torch.arange(many, device=DEV) % few
    got = torch.zeros((many,) + fd.shape[1:], dtype=torch.from_numpy(fd).dtype, device=DEV)
    hydro.interpolate(torch.from_numpy(cd).to(DEV)[at].contiguous(), got, (1, 1, 1), size, **kw)
    assert torch.equal(got, torch.from_numpy(want).to(DEV)[at])
