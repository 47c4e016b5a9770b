"""GPU: the copies between a periodic level and patch groups (gather, scatter, transpose of the gather) over ghost
widths, one to three patch groups per axis, both types, and destinations without vector alignment."""
import numpy as np
import pytest

from gamer_amd import ic

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _unaligned(shape, dtype):
    """A contiguous device tensor whose first element lies one element past an aligned address."""
    n = int(np.prod(shape))
    return torch.full((n + 1,), -7.0, dtype=dtype, device=DEV)[1:].view(shape)


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("ghost", [0, 1, 3, 8])
@pytest.mark.parametrize("shape", [(1, 1, 1), (2, 1, 3), (3, 2, 1)])
def test_level_copies(shape, ghost, dtype):
    from gamer_amd import hydro
    print(f"[gpu] level copies {shape} ghost={ghost} {dtype}", flush=True)
    nz, ny, nx = (16 * k for k in shape)
    rng = np.random.Generator(np.random.PCG64(11))
    cons = rng.standard_normal((5, nz, ny, nx)).astype(np.float64 if dtype == torch.float64 else np.float32)
    want = ic.cut_patch_groups(cons, ghost)
    level = torch.from_numpy(cons).to(DEV)
    for out in (None, _unaligned(want.shape, dtype)):
        got = hydro.prepare_uniform(level, ghost, out=out)
        torch.cuda.synchronize()
        np.testing.assert_array_equal(got.cpu().numpy(), want)
    inner = torch.from_numpy(ic.cut_patch_groups(cons, 0)).to(DEV)
    for dst in (torch.zeros_like(level), _unaligned(tuple(level.shape), dtype)):
        hydro.close_uniform(inner, dst)
        torch.cuda.synchronize()
        np.testing.assert_array_equal(dst.cpu().numpy(), cons)
    # the transpose: sum of every copy of a cell, in double, rounded once
    lam = rng.standard_normal(want.shape).astype(cons.dtype)
    ref = np.zeros(cons.shape)
    i = np.arange(16 + 2 * ghost) - ghost
    for p in range(lam.shape[0]):
        px, py, pz = p % shape[2], (p // shape[2]) % shape[1], p // (shape[2] * shape[1])
        np.add.at(ref, (slice(None), ((pz * 16 + i) % nz)[:, None, None], ((py * 16 + i) % ny)[None, :, None],
                        ((px * 16 + i) % nx)[None, None, :]), lam[p].astype(np.float64))
    got = hydro.prepare_uniform_adjoint(torch.from_numpy(lam).to(DEV), cons.shape, ghost)
    torch.cuda.synchronize()
    eps = np.finfo(cons.dtype).eps                      # 8 terms summed in double, then one rounding
    np.testing.assert_allclose(got.cpu().numpy(), ref, rtol=eps, atol=8 * 4 * np.finfo(np.float64).eps)
