"""GPU: the HLLC interface solve of the marching kernels on states of very different density, face by face.

A time step of 1e-30 leaves the half step without effect, and inputs that are uniform along the face normal on either
side of the middle coarse-fine plane have no slopes there, so the plane's fluxes are those of the input states: one random
Riemann problem per cell of the plane."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu
DEV = "cuda:0"
GAMMA = 5.0 / 3.0
NPG = 4


def _hllc(left, right, d):
    """HLLC flux across a d-normal face between (rho, vx, vy, vz, P) states, in the type of its inputs."""
    cs = [np.sqrt(GAMMA * w[4] / w[0]) for w in (left, right)]
    cons = [np.stack([w[0], w[0] * w[1], w[0] * w[2], w[0] * w[3], w[4] / (np.longdouble(GAMMA) - 1)
                      + w[0] * (w[1] ** 2 + w[2] ** 2 + w[3] ** 2) / 2]) for w in (left, right)]
    ul, ur, pl, pr = left[1 + d], right[1 + d], left[4], right[4]
    wl, wr = np.minimum(ul - cs[0], ur - cs[1]), np.maximum(ul + cs[0], ur + cs[1])
    tl, tr = left[0] * (ul - wl), right[0] * (wr - ur)
    vs = (tl * ul + tr * ur + pl - pr) / (tl + tr)
    ps = (tl * pr + tr * pl + tl * tr * (ul - ur)) / (tl + tr)
    at = vs >= 0
    u, p, sp = np.where(at, ul, ur), np.where(at, pl, pr), np.where(at, np.minimum(wl, 0), np.maximum(wr, 0))
    f = (u - sp) * np.where(at, cons[0], cons[1])
    f[1 + d] += p
    f[4] += u * p
    f *= vs / (vs - sp)
    cp = -sp * ps / (vs - sp)
    f[1 + d] += cp
    f[4] += cp * vs
    return f


def _states(kind, rng, shape):
    """Heavy and light states (velocities along the normal as seen from the heavy side, the light side towards +)."""
    c = 10.0 ** rng.uniform(3.5, 6.0, shape)
    z = np.ones(shape)
    if kind == "flow":         # equal sound speeds 1, both moving into the heavy side's direction, the contact with them
        u = rng.uniform(-0.95, -0.75, shape)
        return (z, u, z / GAMMA), (z / c, u, z / c / GAMMA)
    # a cold light jet (Mach 30 to 300, so no wave speed cancels) onto a slow heavy state that recedes from it
    u, jet, mach = rng.uniform(-0.7, -0.3, shape), rng.uniform(200.0, 400.0, shape), 10.0 ** rng.uniform(1.5, 2.5, shape)
    return (z, u, z / GAMMA), (z / c, u - jet, z / c / GAMMA * (jet / mach) ** 2)


@pytest.mark.parametrize("prec", ["fp32", "fp64"])
@pytest.mark.parametrize("kind", ["flow", "jet"])
@pytest.mark.parametrize("scheme", ["MHM_RP", "MHM"])
def test_light_gas_at_a_heavy_contact(scheme, kind, prec):
    """The contact moves into the heavy side, so the flux is the light gas's.  No component cancels, and no operation of
    the solve takes a rounding of the heavy side's pressure or of the fast side's velocity into it: a chain of about 30
    roundings, taken at their full size one on top of the other, and twice that as the bound, relative to each component."""
    from gamer_amd import hydro
    dtype, n = (np.float32 if prec == "fp32" else np.float64), hydro.NX[scheme]
    g, tol = (n - 16) // 2, 64 * (2.0 ** -24 if prec == "fp32" else 2.0 ** -53)
    for d in range(3):
        for mirrored in (False, True):
            print(f"[gpu] heavy contact {scheme} {kind} {prec} direction {d} mirrored {mirrored}", flush=True)
            rng = np.random.default_rng(31)
            axis = 3 - d                                              # of (npg, z, y, x)
            sides = []
            for rho, u, p in _states(kind, rng, (NPG, n, n)):
                v = [rng.uniform(0.2, 0.4, (NPG, n, n)) for _ in range(3)]
                v[d] = -u if mirrored else u
                e = p / (GAMMA - 1.0) + 0.5 * rho * (v[0] ** 2 + v[1] ** 2 + v[2] ** 2)
                sides.append(np.stack([rho, rho * v[0], rho * v[1], rho * v[2], e], 1).astype(dtype))
            if mirrored:
                sides.reverse()
            half = n // 2
            cells = np.concatenate([np.repeat(np.expand_dims(s, axis + 1), half, axis + 1) for s in sides], axis + 1)
            _, flux = hydro.fluid_solver(torch.from_numpy(np.ascontiguousarray(cells)).to(DEV), 1e-30, 1.0 / 64, scheme=scheme)
            got = flux.cpu().numpy()[:, 3 * d + 1]                    # (npg, 5, 16, 16)
            prim = []
            for s in sides:
                c = [q.astype(np.longdouble)[:, g:g + 16, g:g + 16] for q in s.transpose(1, 0, 2, 3)]
                k = (c[1] ** 2 + c[2] ** 2 + c[3] ** 2) / (2 * c[0])
                prim.append(np.stack([c[0], c[1] / c[0], c[2] / c[0], c[3] / c[0], (np.longdouble(GAMMA) - 1) * (c[4] - k)]))
            want = _hllc(*prim, d).transpose(1, 0, 2, 3)
            err = (np.abs(got - want) / np.abs(want)).max(axis=(0, 2, 3))
            assert (err <= tol).all(), (d, mirrored, (err / tol).astype(float))


@pytest.mark.parametrize("contrast", [1e2, 1e4, 1e6])
@pytest.mark.parametrize("scheme", ["MHM_RP", "MHM"])
def test_light_cells_beside_heavy_gas_after_a_step(scheme, contrast):
    """The same flow through a whole FP32 step, half step included, against the FP64 oracle on the same inputs, every cell
    relative to itself (momenta to sqrt(rho E)): two flux errors of 64 half ulps times dt/dh (|u| + c) = 0.3, and the
    roundings of the states the fluxes start from, are well below 128 half ulps."""
    import oracle
    from gamer_amd import hydro
    n, tol = hydro.NX[scheme], 128 * 2.0 ** -24
    dh = 1.0 / 64
    dt = 0.3 * dh / 1.9
    for d in range(3):
        for mirrored in (False, True):
            print(f"[gpu] step at a heavy contact {scheme} {contrast:g} direction {d} mirrored {mirrored}", flush=True)
            heavy = np.arange(n) < n // 2
            heavy = heavy[::-1] if mirrored else heavy
            rho = np.where(heavy, 1.0, 1.0 / contrast)
            v = np.zeros((3, n))
            v[d] = 0.9 if mirrored else -0.9
            line = np.stack([rho, *(rho * v), rho / GAMMA / (GAMMA - 1.0) + 0.5 * rho * 0.81])
            shape = [1, 5, 1, 1, 1]
            shape[4 - d] = n
            u = np.ascontiguousarray(np.broadcast_to(line.reshape(shape), (1, 5, n, n, n)).astype(np.float32))
            out, _ = hydro.fluid_solver(torch.from_numpy(u).to(DEV), dt, dh, scheme=scheme)
            want, _ = oracle.fluid_solver(u.astype(np.float64), dt, dh, scheme=scheme)
            got, scale = out.cpu().numpy(), np.abs(want)
            scale[:, 1:4] = np.sqrt(want[:, :1] * want[:, 4:])
            err = (np.abs(got - want) / scale).max(axis=(0, 2, 3, 4))
            assert (err <= tol).all(), (d, mirrored, (err / tol).astype(float))
