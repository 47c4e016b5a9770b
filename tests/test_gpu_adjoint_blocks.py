"""GPU: the adjoint and tangent kernels in blocks of one plane (few patch groups) and in marching blocks (many)."""
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("rsolver", ["HLLC", "HLLE", "ROE"])
def test_few_and_many_groups_give_the_same_bits(rsolver):
    """140 patch groups march on 256 compute units, parts of 1, 47, 48, 60 and 63 of them do not in one phase or the other;
    every face and cell is computed alike."""
    from gamer_amd import hydro
    print(f"[gpu] adjoint and tangent blocks {rsolver}", flush=True)
    g = torch.Generator(device=DEV).manual_seed(37)
    r = torch.rand((140, 5, 22, 22, 22), dtype=torch.float64, device=DEV, generator=g)
    u = r.clone()
    u[:, 0] = 0.5 + r[:, 0]
    u[:, 1:4] = u[:, :1] * (r[:, 1:4] - 0.5)
    u[:, 4] = 1.0 + r[:, 4] + 0.5 * (u[:, 1:4] ** 2).sum(1) / u[:, 0]
    lam = torch.randn((140, 5, 16, 16, 16), dtype=torch.float64, device=DEV, generator=g)
    tan = torch.randn(u.shape, dtype=torch.float64, device=DEV, generator=g)
    a = hydro.mhm_adjoint(u, lam, 2e-3, 1.0 / 64, rsolver=rsolver)
    out, jv = hydro.mhm_tangent(u, tan, 2e-3, 1.0 / 64, rsolver=rsolver)
    assert torch.isfinite(a).all() and torch.isfinite(jv).all()
    for at in (slice(0, 1), slice(1, 48), slice(48, 96), slice(80, 140), slice(30, 93)):
        assert torch.equal(hydro.mhm_adjoint(u[at], lam[at], 2e-3, 1.0 / 64, rsolver=rsolver), a[at]), at
        o, j = hydro.mhm_tangent(u[at], tan[at], 2e-3, 1.0 / 64, rsolver=rsolver)
        assert torch.equal(o, out[at]) and torch.equal(j, jv[at]), at
