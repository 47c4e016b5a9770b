"""GPU: the marching solver kernels (hydro_mhm_rp.hip, hydro_mhm.hip) where their forms could go wrong."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("rsolver", ["HLLE", "ROE"])
@pytest.mark.parametrize("scheme", ["MHM_RP", "MHM"])
def test_cold_uniform_flow_is_a_fixed_point(scheme, rsolver, prec):
    """Zero pressure, so zero sound speed: HLLE's wave speeds coincide across the flow, Roe's squared sound speed is 0
    and every face is supersonic.  rho = 1, v = (1, 0, 0), E = 1/2 are exact, and so are the upwind fluxes."""
    from gamer_amd import hydro
    print(f"[gpu] cold uniform flow {scheme} {rsolver} {prec}", flush=True)
    dtype, n = (np.float64 if prec == "fp64" else np.float32), (22 if scheme == "MHM_RP" else 20)
    g = (n - 16) // 2
    u = np.zeros((2, 5, n, n, n), dtype=dtype)
    u[:, 0], u[:, 1], u[:, 4] = 1.0, 1.0, 0.5
    out, flux = hydro.fluid_solver(torch.from_numpy(u).to(DEV), 0.01, 1.0 / 64, scheme=scheme, rsolver=rsolver)
    torch.cuda.synchronize()
    f = flux.cpu().numpy()
    np.testing.assert_array_equal(out.cpu().numpy(), u[:, :, g:g + 16, g:g + 16, g:g + 16])
    want = np.array([1.0, 1.0, 0.0, 0.0, 0.5], dtype=dtype)[None, None, :, None, None]
    np.testing.assert_array_equal(f[:, 0:3], np.broadcast_to(want, f[:, 0:3].shape))
    np.testing.assert_array_equal(f[:, 3:9], 0.0)


def _random_groups(npg, n, dtype):
    """Patch groups of admissible gas with contrasts in every field, drawn on the device."""
    g = torch.Generator(device=DEV).manual_seed(20)
    r = torch.rand((npg, 5, n, n, n), dtype=dtype, device=DEV, generator=g)
    u = r.clone()
    u[:, 0] = 0.5 + r[:, 0]
    u[:, 1:4] = u[:, :1] * (r[:, 1:4] - 0.5)
    u[:, 4] = 1.0 + r[:, 4] + 0.5 * (u[:, 1:4] ** 2).sum(1) / u[:, 0]
    return u


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("rsolver,limiter,store_flux,with_dt", [
    ("HLLC", "VL_GMINMOD", True, False), ("ROE", "VANLEER", True, True), ("HLLE", "GMINMOD", False, True)])
@pytest.mark.parametrize("scheme", ["MHM_RP", "MHM"])
def test_slabs_equal_whole_groups(scheme, rsolver, limiter, store_flux, with_dt, prec):
    """The launch splits what does not fill the chip into z slabs.  1024 patch groups fill it with whole ones on 256 compute
    units (one or two groups each); every smaller call has to give the same bits, fluxes and time steps included, and the
    work queue, which never splits, too."""
    from gamer_amd import hydro
    print(f"[gpu] slabs {scheme} {rsolver} {limiter} flux {store_flux} dt {with_dt} {prec}", flush=True)
    dtype = torch.float64 if prec == "fp64" else torch.float32
    u = _random_groups(1024, hydro.NX[scheme], dtype)
    g = torch.Generator(device=DEV).manual_seed(21)
    dtdh = torch.rand((1024, 2), dtype=torch.float64, device=DEV, generator=g) * 1e-4 + 1e-4
    dtdh[:, 1] = 1.0 / 64

    def solve(n, **kw):
        dtp = torch.full((n, 8), -1.0, dtype=dtype, device=DEV) if with_dt else None
        out, flux = hydro.solve_batch(u[:n], dtdh[:n], scheme=scheme, rsolver=rsolver, limiter=limiter, store_flux=store_flux,
                                      dt_patch=dtp, **kw)
        return [x for x in (out, flux, dtp) if x is not None]

    whole = solve(1024)
    queue = solve(1024, queue_counter=torch.zeros(1, dtype=torch.int32, device=DEV), groups_per_cu=1)
    for w, q in zip(whole, queue):
        assert torch.isfinite(w).all()
        assert torch.equal(w, q)
    for n in (1, 3, 17, 40, 100, 130, 260, 300, 513, 700):
        for w, s in zip(whole, solve(n)):
            assert torch.equal(w[:n], s), n


def test_retry_is_decided_over_the_whole_group():
    """The MinMod retry redoes a patch group where any of its cells fails, so such calls are not split: three groups, one
    with a cell that fails for every coefficient, equal the same groups among 1024."""
    from gamer_amd import hydro
    print("[gpu] minmod retry, few groups", flush=True)
    u = _random_groups(1024, 22, torch.float64)
    u[1, 4, 11, 11, 18] = 400.0
    kw = dict(limiter="GMINMOD", minmod_maxiter=2)
    whole, _ = hydro.fluid_solver(u, 2e-2, 1.0 / 64, **kw)
    few, _ = hydro.fluid_solver(u[:3], 2e-2, 1.0 / 64, **kw)
    assert torch.equal(whole[:3].view(torch.int64), few.view(torch.int64))
