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
