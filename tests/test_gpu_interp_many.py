"""GPU: interpolation of many boxes, whose launches differ from those of a few in lanes and form: the same bits."""
import numpy as np
import pytest

import oracle

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("scheme", ["MINMOD3D", "MINMOD1D", "VANLEER", "CQUAD", "QUAD", "CQUAR", "QUAR"])
@pytest.mark.parametrize("opts", [{}, {"opp_sign_0th": True}, {"monotonic": 0x0B}])
def test_many_boxes_equal_few(opts, scheme, dtype):
    """Steep contrasts, so that some boxes take the retries; the first boxes also against the oracle without them."""
    from gamer_amd import hydro
    print(f"[gpu] many boxes {scheme} {opts} {dtype}", flush=True)
    g = 2 if scheme in ("CQUAR", "QUAR") else 1
    red = scheme in ("CQUAD", "QUAD", "CQUAR", "QUAR")
    rng = torch.Generator(device=DEV).manual_seed(43)
    for nbox, cr, masked in ((600, (4, 4, 4), False), (600, (6, 5, 7), False), (600, (12, 11, 10), False), (513, (16, 16, 8), False),
                             (1100, (8, 7, 8), True)):
        n = tuple(c + 2 * g for c in reversed(cr))
        c = torch.rand((nbox, 5) + n, dtype=torch.float64, device=DEV, generator=rng)
        c[:, 0] = 10.0 ** (2.0 * c[:, 0] - 1.0)
        c[:, 1:4] = c[:, :1] * 6.0 * (c[:, 1:4] - 0.5)
        c[:, 4] = 0.01 + c[:, 4] + 0.5 * (c[:, 1:4] ** 2).sum(1) / c[:, 0]
        c = c.to(dtype)
        fine = tuple(2 * k for k in reversed(cr))
        need = (torch.rand((nbox,) + tuple(reversed(cr)), device=DEV, generator=rng) < 0.4).to(torch.uint8) if masked else None

        def run(at, **kw):
            cc, f = c[at].clone(), torch.full((len(range(*at.indices(nbox))), 5) + fine, -3.0, dtype=dtype, device=DEV)
            bad = hydro.interpolate(cc, f, (g,) * 3, cr, scheme=scheme, need=need[at].contiguous() if masked else None, **opts, **kw)
            return cc, f, int(bad.item())

        for kw in (dict(int_prim=False, reduce_mono=False), dict(reduce_mono=red)):
            many = run(slice(0, nbox), **kw)
            few = [run(slice(i, min(i + 90, nbox)), **kw) for i in range(0, nbox, 90)]
            assert torch.equal(many[0], torch.cat([x[0] for x in few])), (nbox, cr, kw)
            assert torch.equal(many[1], torch.cat([x[1] for x in few])), (nbox, cr, kw)
            assert many[2] == sum(x[2] for x in few)
        if not masked:
            fd = np.full((4, 5) + fine, -3.0, dtype=c.cpu().numpy().dtype)
            _, want, _ = oracle.interpolate(c[:4].cpu().numpy(), fd, (g,) * 3, cr, scheme=scheme, int_prim=False, reduce_mono=False, **opts)
            np.testing.assert_array_equal(run(slice(0, nbox), int_prim=False, reduce_mono=False)[1][:4].cpu().numpy(), want)
