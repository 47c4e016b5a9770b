"""GPU: a small and a large host-array call of several streams, one after the other without a wait between them."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("large_first", [True, False])
@pytest.mark.parametrize("nstream", [2, 3, 4])
def test_small_and_large_calls_share_the_device_arrays(nstream, large_first):
    """The small call has groups on every stream, so the large one waits for all of them (or they for it)."""
    from gamer_amd import hydro
    print(f"[gpu] host call order {nstream} streams, large first {large_first}", flush=True)
    large, small, dh = 60, 5 * nstream + 1, 1.0 / 64
    g = torch.Generator(device=DEV).manual_seed(29)
    sets = []
    for n in (large, small) if large_first else (small, large):
        r = torch.rand((n, 5, 22, 22, 22), dtype=torch.float64, device=DEV, generator=g)
        r[:, 0] += 0.5
        r[:, 1:4] = r[:, :1] * (r[:, 1:4] - 0.5)
        r[:, 4] += 1.0 + 0.5 * (r[:, 1:4] ** 2).sum(1) / r[:, 0]
        sets.append([x.cpu().numpy() for x in (r, *hydro.fluid_solver(r, 1e-3, dh))])
    api = hydro.GpuFluidApi(large, gpu_nstream=nstream, precision="fp64")
    try:
        for _ in range(3):
            for k, (u, _, _) in enumerate(sets):
                h_in, h_out, h_flux = api.host_arrays(k)
                h_in[:len(u)] = u
                h_out[:] = h_flux[:] = -1.0
            for k, (u, _, _) in enumerate(sets):
                api.asyn_fluid_solver(k, len(u), 1e-3, dh)
            api.synchronize()
            for k, (u, out, flux) in enumerate(sets):
                _, h_out, h_flux = api.host_arrays(k)
                np.testing.assert_array_equal(h_out[:len(u)], out)
                np.testing.assert_array_equal(h_flux[:len(u)], flux)
                assert (h_out[len(u):] == -1.0).all()
    finally:
        api.free()
