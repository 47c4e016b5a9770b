"""GPU: host-array calls large enough to be cut into pieces with both copy directions in flight, against the device call,
one after the other without a wait and mixed with small ones."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("precision,npg,nstream", [("fp64", 50, 1), ("fp64", 97, 4), ("fp32", 100, 3)])
@pytest.mark.parametrize("store_flux", [True, False])
def test_large_host_calls(store_flux, precision, npg, nstream):
    from gamer_amd import hydro
    print(f"[gpu] large host calls {precision} {npg} {nstream} flux {store_flux}", flush=True)
    dtype = torch.float64 if precision == "fp64" else torch.float32
    g = torch.Generator(device=DEV).manual_seed(23)
    kw = dict(store_flux=store_flux, rsolver="HLLC")
    sets, dh = [], 1.0 / 64
    for k in range(2):
        r = torch.rand((npg, 5, 22, 22, 22), dtype=dtype, device=DEV, generator=g)
        u = r.clone()
        u[:, 0] = 0.5 + r[:, 0]
        u[:, 1:4] = u[:, :1] * (r[:, 1:4] - 0.5)
        u[:, 4] = 1.0 + r[:, 4] + 0.5 * (u[:, 1:4] ** 2).sum(1) / u[:, 0]
        sets.append([x.cpu().numpy() if x is not None else None for x in (u, *hydro.fluid_solver(u, 1e-3, dh, **kw))])
    api = hydro.GpuFluidApi(npg, gpu_nstream=nstream, precision=precision)
    try:
        # one stream keeps calls of any size in order; several only calls of one size, so the small one waits there
        for order in ((npg, npg), (npg, 2), (2, npg)):
            for k, n in enumerate(order):
                h_in, h_out, h_flux = api.host_arrays(k)
                h_in[:n] = sets[k][0][:n]
                h_out[:] = -1.0
                h_flux[:] = -1.0
            for k, n in enumerate(order):
                api.asyn_fluid_solver(k, n, 1e-3, dh, **kw)
                if nstream > 1 and order[0] != order[1]:
                    api.synchronize()
            api.synchronize()
            for k, n in enumerate(order):
                _, h_out, h_flux = api.host_arrays(k)
                np.testing.assert_array_equal(h_out[:n], sets[k][1][:n])
                assert (h_out[n:] == -1.0).all()
                if store_flux:
                    np.testing.assert_array_equal(h_flux[:n], sets[k][2][:n])
                else:
                    assert (h_flux == -1.0).all()
    finally:
        api.free()
