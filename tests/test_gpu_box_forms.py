"""GPU: the box gather in blocks across boxes (small ones), by chunks and by planes (large ones), against the oracle."""
import numpy as np
import pytest

import oracle

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("nbox,size,origin", [(700, (3, 5, 2), (6, 4, 7)), (5, (8, 8, 8), (0, 3, 7)), (300, (9, 8, 7), (2, 2, 1)),
                                              (40, (24, 24, 24), (5, 6, 7)), (60, (30, 19, 27), (1, 0, 3))])
def test_box_forms(nbox, size, origin, dtype):
    from gamer_amd import hydro
    print(f"[gpu] box gather {nbox} x {size} {dtype.__name__}", flush=True)
    rng = np.random.default_rng(47)
    patch, late = rng.standard_normal((2, 29, 5, 8, 8, 8)).astype(dtype)
    tdim = tuple((o + n + 7) // 8 for o, n in zip(origin, size))
    slot = rng.integers(-4, 29, (nbox,) + tdim[::-1]).clip(-1).astype(np.int32)
    box = np.full((nbox, 5) + size[::-1], -6.0, dtype=dtype)
    T = lambda a: torch.from_numpy(a).to(DEV)  # noqa: E731
    got = T(box.copy())
    hydro.gather_boxes(T(patch), got, T(slot), origin)
    np.testing.assert_array_equal(got.cpu().numpy(), oracle.gather_boxes(patch, box, slot, origin))
    got = T(box.copy())
    hydro.gather_boxes(T(patch), got, T(slot), origin, mean_with=T(late))
    np.testing.assert_array_equal(got.cpu().numpy(), oracle.gather_boxes((patch + late) * dtype(0.5), box, slot, origin))
