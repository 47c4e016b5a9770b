"""GPU: interpolation of the asked-for coarse cells and the copies around it where their forms could go wrong: few, many
and no cells, cell counts off the block size, general monotonic and clipping options, ghost widths and box sizes."""
import numpy as np
import pytest

import oracle

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _gas(rng, shape, dtype):
    """Conserved fields with steep contrasts: some interpolated cells are unphysical and take the retries."""
    u = rng.random(shape)
    u[:, 0] = 10.0 ** (2.0 * u[:, 0] - 1.0)
    u[:, 1:4] = u[:, :1] * 6.0 * (u[:, 1:4] - 0.5)
    u[:, 4] = 0.01 + u[:, 4] + 0.5 * (u[:, 1:4] ** 2).sum(1) / u[:, 0]
    return u.astype(dtype)


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("scheme", ["MINMOD3D", "MINMOD1D", "VANLEER", "CQUAD", "QUAD", "CQUAR", "QUAR"])
@pytest.mark.parametrize("opts", [{}, {"monotonic": 0x0B}, {"opp_sign_0th": True}])
def test_asked_for_cells(scheme, opts, dtype):
    from gamer_amd import hydro
    print(f"[gpu] masks {scheme} {opts} {dtype.__name__}", flush=True)
    rng = np.random.Generator(np.random.PCG64(5))
    g = 2 if scheme in ("CQUAR", "QUAR") else 1
    cr = (12, 11, 9)                                            # x, y, z: 1188 cells
    n, nbox = tuple(c + 2 * g for c in reversed(cr)), 6
    cd = _gas(rng, (nbox, 5) + n, dtype)
    need = np.zeros((nbox, 9, 11, 12), dtype=np.uint8)          # box 0: none
    need[1, 4, 5, 6] = 1
    need[2, :2] = 1
    need[3, :, :, 10:] = 1
    need[4] = rng.random(need[4].shape) < 0.6
    need[5] = 1
    fd = np.full((nbox, 5) + tuple(2 * c for c in reversed(cr)), -3.0, dtype=dtype)
    _, want, _ = oracle.interpolate(cd, fd, (g,) * 3, cr, scheme=scheme, int_prim=False, reduce_mono=False, **opts)
    keep = np.repeat(np.repeat(np.repeat(need, 2, 1), 2, 2), 2, 3)[:, None] == 0
    got = torch.from_numpy(fd.copy()).to(DEV)
    hydro.interpolate(torch.from_numpy(cd).to(DEV), got, (g,) * 3, cr, scheme=scheme, int_prim=False, reduce_mono=False,
                      need=torch.from_numpy(need).to(DEV), **opts)
    np.testing.assert_array_equal(got.cpu().numpy(), np.where(keep, dtype(-3.0), want))
    # with the retries, every cell asked for: as the oracle, whose arithmetic is the same
    opts = dict(opts, reduce_mono=scheme in ("CQUAD", "QUAD", "CQUAR", "QUAR"))
    cw, want, nf = oracle.interpolate(cd, fd, (g,) * 3, cr, scheme=scheme, **opts)
    c, got = torch.from_numpy(cd).to(DEV), torch.from_numpy(fd.copy()).to(DEV)
    n_bad = hydro.interpolate(c, got, (g,) * 3, cr, scheme=scheme, **opts)
    tol = dict(rtol=64 * np.finfo(dtype).eps, atol=64 * np.finfo(dtype).eps * np.abs(want).max())
    assert int(n_bad.item()) == nf
    np.testing.assert_allclose(c.cpu().numpy(), cw, **tol)
    if nf == 0:                                                 # the cells that stay unphysical have no defined value
        np.testing.assert_allclose(got.cpu().numpy(), want, **tol)


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("ghost", [0, 1, 3, 8])
def test_windows_and_boxes(ghost, dtype):
    from gamer_amd import hydro
    print(f"[gpu] windows and boxes ghost {ghost} {dtype.__name__}", flush=True)
    rng = np.random.Generator(np.random.PCG64(6))
    npatch, npg, n = 37, 3, 16 + 2 * ghost
    patch = rng.standard_normal((npatch, 5, 8, 8, 8)).astype(dtype)
    slot = rng.integers(-8, npatch, (npg, 4, 4, 4)).clip(-1).astype(np.int32)
    fb = rng.standard_normal((npg, 5, n + 3, n + 2, n + 1)).astype(dtype)
    T = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(DEV)
    pg = np.full((npg, 5, n, n, n), -5.0, dtype=dtype)
    flat = torch.full((pg.size + 1,), -5.0, dtype=T(pg).dtype, device=DEV)
    for dst in (T(pg), flat[1:].view(pg.shape)):               # aligned, and one element past it
        hydro.prepare_patches(T(patch), dst, T(slot), ghost)
        np.testing.assert_array_equal(dst.cpu().numpy(), oracle.prepare_patches(patch, pg, slot, ghost))
        hydro.assemble_patch_groups(T(patch), T(fb), dst, T(slot), ghost, (1, 2, 3))
        np.testing.assert_array_equal(dst.cpu().numpy(), oracle.assemble_patch_groups(patch, fb, pg, slot, ghost, (1, 2, 3)))
    for size, origin, tdim in (((1, 1, 1), (0, 0, 0), (1, 1, 1)), ((14, 14, 14), (5, 5, 5), (3, 3, 3)),
                               ((33, 7, 19), (6, 1, 4), (5, 1, 3)), ((16, 16, 6), (0, 0, 10), (2, 2, 2)),
                               ((128, 64, 128), (0, 3, 5), (16, 9, 17)), ((101, 103, 101), (1, 0, 2), (13, 13, 13))):
        bs = rng.integers(-4, npatch, (npg,) + tdim[::-1]).clip(-1).astype(np.int32)
        box = np.full((npg, 5) + size[::-1], -6.0, dtype=dtype)
        dst = T(box)
        hydro.gather_boxes(T(patch), dst, T(bs), origin)
        np.testing.assert_array_equal(dst.cpu().numpy(), oracle.gather_boxes(patch, box, bs, origin))
        late = rng.standard_normal(patch.shape).astype(dtype)
        dst = T(box)
        hydro.gather_boxes(T(patch), dst, T(bs), origin, mean_with=T(late))
        np.testing.assert_array_equal(dst.cpu().numpy(), oracle.gather_boxes((patch + late) * dtype(0.5), box, bs, origin))
