"""GPU: conservative quadratic interpolation at monotonic coefficients off the usual 1 to 4, against the oracle."""
import numpy as np
import pytest

import oracle

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("monotonic", [0x1F, 0x15])
@pytest.mark.parametrize("coeff", [-1.5, 0.0, 0.4, 1.0, 7.0])
def test_cquad_coefficients(coeff, monotonic, dtype):
    """The slope is the smallest of three signed values, so a coefficient below 0 turns it around: the same operations in
    the same order as the oracle, and the same bits."""
    from gamer_amd import hydro
    print(f"[gpu] cquad coefficient {coeff} monotonic {monotonic:#x} {dtype.__name__}", flush=True)
    cd = np.random.default_rng(41).standard_normal((3, 5, 9, 8, 7)).astype(dtype)
    fd = np.zeros((3, 5, 14, 12, 10), dtype=dtype)
    kw = dict(scheme="CQUAD", mono_coeff=coeff, monotonic=monotonic, int_prim=False, reduce_mono=False)
    _, want, _ = oracle.interpolate(cd, fd, (1, 1, 1), (5, 6, 7), **kw)
    got = torch.from_numpy(fd).to(DEV)
    hydro.interpolate(torch.from_numpy(cd).to(DEV), got, (1, 1, 1), (5, 6, 7), **kw)
    np.testing.assert_array_equal(got.cpu().numpy(), want)
