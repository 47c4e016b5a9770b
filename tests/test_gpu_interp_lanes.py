"""GPU: interpolation calls at the edges between the numbers of lanes and the forms that a call can take, against the oracle."""
import numpy as np
import pytest

import oracle

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("scheme", ["MINMOD3D", "MINMOD1D", "VANLEER", "CQUAD", "QUAD", "CQUAR", "QUAR"])
@pytest.mark.parametrize("masked", [False, True])
def test_lanes_and_forms(masked, scheme, dtype):
    """Boxes of 64, 65, 128, 132, 256, 270 and 800 cells; of 32, 33, 64, 65, 128 and 130 columns; thin ones; few boxes, from
    two, three and eight per compute unit on: the same operations in the same order as the oracle, and the same bits."""
    from gamer_amd import hydro
    print(f"[gpu] interpolation lanes {scheme} masked {masked} {dtype.__name__}", flush=True)
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    g, rng, few = (2 if scheme in ("CQUAR", "QUAR") else 1), np.random.default_rng(49), 3
    for size in ((8, 8, 1), (13, 5, 1), (8, 4, 4), (11, 3, 4), (8, 8, 2), (11, 12, 1), (16, 16, 1), (9, 6, 5), (13, 5, 4), (16, 8, 5), (13, 10, 6),
                 (10, 10, 8), (16, 16, 2)):
        cd = rng.standard_normal((few, 5) + tuple(n + 2 * g for n in reversed(size))).astype(dtype)
        fd = np.full((few, 5) + tuple(2 * n for n in reversed(size)), -3.0, dtype=dtype)
        need = (rng.random((few,) + size[::-1]) < 0.4).astype(np.uint8) if masked else None
        for opts in ({}, {"opp_sign_0th": True, "monotonic": 0x15}):
            kw = dict(scheme=scheme, int_prim=False, reduce_mono=False, **opts)
            _, want, _ = oracle.interpolate(cd, fd, (g,) * 3, size, **kw)
            if masked:
                keep = np.repeat(np.repeat(np.repeat(need, 2, 1), 2, 2), 2, 3)[:, None] == 0
                want = np.where(keep, fd, want)
            want = torch.from_numpy(want).to(DEV)
            for nbox in (few, 2 * cus, 3 * cus, 8 * cus):
                at = torch.arange(nbox, device=DEV) % few
                got = torch.from_numpy(fd).to(DEV)[at].contiguous()
                m = {"need": torch.from_numpy(need).to(DEV)[at].contiguous()} if masked else {}
                hydro.interpolate(torch.from_numpy(cd).to(DEV)[at].contiguous(), got, (g,) * 3, size, **kw, **m)
                assert torch.equal(got, want[at]), (size, opts, nbox)
