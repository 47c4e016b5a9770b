"""GPU: the adjoint's kernels at the edges of their row and plane blocks: single entries of J^T lambda against the tangent
of the same unit input."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("limiter", ["VL_GMINMOD", "VANLEER"])
@pytest.mark.parametrize("rsolver", ["HLLC", "HLLE", "ROE"])
def test_entries_against_unit_tangents(rsolver, limiter):
    from gamer_amd import hydro
    print(f"[gpu] adjoint entries {rsolver} {limiter}", flush=True)
    rng = np.random.Generator(np.random.PCG64(17))
    # the diagonal, the middles of the faces of the block of cells, and cells at random
    cells = [(a, a, a) for a in range(22)]
    for a in range(22):
        cells += [(a, 10, 11), (11, a, 10), (10, 11, a)]
    cells += [tuple(rng.integers(0, 22, 3)) for _ in range(112)]
    npg = len(cells)
    g = torch.Generator(device=DEV).manual_seed(18)
    r = torch.rand((1, 5, 22, 22, 22), dtype=torch.float64, device=DEV, generator=g)
    u = r.clone()
    u[:, 0] = 0.7 + 0.6 * r[:, 0]
    u[:, 1:4] = u[:, :1] * 1.5 * (r[:, 1:4] - 0.4)
    u[:, 4] = 1.0 + 0.6 * r[:, 4] + 0.5 * (u[:, 1:4] ** 2).sum(1) / u[:, 0]
    u = u.expand(npg, -1, -1, -1, -1).contiguous()
    v = torch.zeros_like(u)
    for p, (k, j, i) in enumerate(cells):
        v[p, p % 5, k, j, i] = 1.0
    lam = torch.randn((npg, 5, 16, 16, 16), dtype=torch.float64, device=DEV, generator=g)
    kw = dict(rsolver=rsolver, limiter=limiter)
    _, jv = hydro.mhm_tangent(u, v, 2e-3, 1.0 / 64, **kw)
    lin = hydro.mhm_adjoint(u, lam, 2e-3, 1.0 / 64, **kw)
    terms = (lam * jv).reshape(npg, -1).cpu().numpy()
    got = (lin * v).reshape(npg, -1).sum(1).cpu().numpy()
    # both sides round each of a few hundred operations a path once; slopes' reciprocals amplify that by their contrast
    np.testing.assert_array_less(np.abs(got - terms.sum(1)), 1e-10 * np.abs(terms).sum(1) + 1e-300)
    assert (np.abs(terms).sum(1) > 0).sum() > npg // 2
