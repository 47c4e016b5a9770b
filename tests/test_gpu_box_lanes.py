"""GPU: the box gather at the edges between its forms (blocks across boxes, by planes, coordinates in double precision)."""
import numpy as np
import pytest

import oracle

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("nbox,size,origin", [(3, (7, 73, 130), (1, 2, 3)), (3, (16, 32, 130), (4, 0, 7)), (90, (33, 31, 5), (2, 3, 1)),
                                              (100, (32, 32, 4), (0, 5, 6)), (1, (8, 17, 8000), (3, 1, 2)), (2, (104, 101, 100), (7, 6, 5))])
def test_box_lanes(nbox, size, origin, dtype):
    """Planes of 511, 512, 1023 and 1024 cells; boxes of more than 2^20 cells."""
    from gamer_amd import hydro
    print(f"[gpu] box gather {nbox} x {size} {dtype.__name__}", flush=True)
    rng = np.random.default_rng(50)
    patch = rng.standard_normal((37, 5, 8, 8, 8)).astype(dtype)
    tdim = tuple((o + n + 7) // 8 for o, n in zip(origin, size))
    slot = rng.integers(-4, 37, (nbox,) + tdim[::-1]).clip(-1).astype(np.int32)
    box = np.full((nbox, 5) + size[::-1], -6.0, dtype=dtype)
    got = torch.from_numpy(box).to(DEV)
    hydro.gather_boxes(torch.from_numpy(patch).to(DEV), got, torch.from_numpy(slot).to(DEV), origin)
    np.testing.assert_array_equal(got.cpu().numpy(), oracle.gather_boxes(patch, box, slot, origin))


def test_more_cells_than_one_launch_holds():
    from gamer_amd import hydro
    nbox, (nx, ny, nz) = 4310, (20, 20, 1000)                          # 8.62e9 cells, one launch holds 8.59e9
    print(f"[gpu] box gather {nbox} x ({nx}, {ny}, {nz})", flush=True)
    gen = torch.Generator(device=DEV).manual_seed(51)
    patch = torch.rand((11, 5, 8, 8, 8), device=DEV, generator=gen)
    slot = torch.randint(0, 11, (nbox, 125, 3, 3), dtype=torch.int32, device=DEV, generator=gen)
    box = torch.empty((nbox, 5, nz, ny, nx), device=DEV)
    hydro.gather_boxes(patch, box, slot, (1, 2, 0))
    for q in (0, 1073, 2147, 4293, 4294, 4295, nbox - 1):
        want = patch[slot[q].long()].permute(3, 0, 4, 1, 5, 2, 6).reshape(5, 1000, 24, 24)[:, :, 2:22, 1:21]
        assert torch.equal(box[q], want), q
