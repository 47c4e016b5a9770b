"""GPU: the transpose of the ghost-zone copies on thin and on full levels, whose launches differ."""
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("ghost", [2, 3, 8])
@pytest.mark.parametrize("shape", [(1, 1, 1), (32, 1, 1), (1, 3, 2), (1, 2, 3), (1, 1, 9), (1, 1, 33), (4, 4, 4), (5, 4, 5)])
def test_transposed_copies(shape, ghost, dtype):
    """Whole-number adjoints, so that the sums are exact in any order: each level cell holds the sum of its copies, which a
    level of its own cell numbers, copied the other way, points out."""
    from gamer_amd import hydro
    print(f"[gpu] transposed level copies {shape} ghost={ghost} {dtype}", flush=True)
    size = (5,) + tuple(16 * k for k in shape)
    cell = torch.arange(torch.Size(size).numel(), dtype=torch.float64, device=DEV).view(size)
    at = hydro.prepare_uniform(cell, ghost).long().flatten()
    g = torch.Generator(device=DEV).manual_seed(53)
    lam = torch.randint(-1000, 1001, (at.numel(),), generator=g, device=DEV)
    want = torch.zeros(cell.numel(), dtype=torch.int64, device=DEV).index_add_(0, at, lam)
    n = 16 + 2 * ghost
    got = hydro.prepare_uniform_adjoint(lam.to(dtype).view(-1, 5, n, n, n), size, ghost)
    assert torch.equal(got.double().flatten(), want.double())
