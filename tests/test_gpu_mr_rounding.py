"""The adaptive P2G weights and the end of RK3, rounding by rounding.  Results
of a step follow these roundings through a solve that stops at a tolerance, so
which products are fused is part of what the kernels compute: the weights of
eq. (6) and the RK3 sum against the same operations on the host."""
import ctypes
from importlib import import_module

import numpy as np
import pytest

from conftest import load_pkg

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu
F = np.float32


def fma(a, b, c):
    """a b + c rounded once: the product of two floats is exact in the 64 bits
    of a long double, and so is the sum but for terms 2^16 apart or more, where
    rounding twice can differ in one case of 2^40."""
    L = np.longdouble
    return (L(a) * L(b) + L(c)).astype(F)


@pytest.mark.parametrize("sorted_", [True, False])
@pytest.mark.parametrize("level", [0, 1])
def test_p2g_weights(sorted_, level):
    """Sums of one particle per support: every sum is one weight, bit for bit."""
    pf = load_pkg()
    cfgm, mrs = (import_module(pf.__name__ + "." + m) for m in ("config", "mr_sim"))
    print(f"[gpu] P2G weights sorted={sorted_} level={level}", flush=True)
    n0, nb = 8, (4, 3, 5)
    dx = 0.37 / n0
    cfg = cfgm.Config(res=tuple(n * n0 for n in nb), dx=dx, ppc=27, droplets=False)
    sim = mrs.AdaptiveSimulator(cfg, nb, n0=n0, max_level=1, frozen_levels=np.full(int(np.prod(nb)), level))
    rng = np.random.default_rng(2)
    # one particle near the middle of each block: supports do not meet
    h = F(dx) * F(1 << level)
    mid = (np.stack(np.meshgrid(*[np.arange(n) for n in nb], indexing="ij"), -1).reshape(-1, 3) + 0.5) * n0 * dx
    x = (mid + rng.uniform(-1, 1, mid.shape) * dx).astype(F)
    sim.set_particles(x, np.zeros_like(x), np.ones(len(x), np.int32), np.full(len(x), level, np.int32))
    sim._rebuild_grid(1e-3)
    prm = sim._params(1e-3, 1.0)
    sim.p2g_sorted = sorted_
    sim.stage_p2g(prm)
    centre = sim.grid.geometry()[0].cpu().numpy()
    weight, mass = sim.cwsum.cpu().numpy(), sim.fmass.cpu().numpy().reshape(-1, 3)
    r = F(cfg.r_p) * F(1 << level)
    inv = F(1) / (r * r)
    bext = F(n0) * F(dx)
    half = F(0.5) * h
    mp = F(cfg.rho_l) * F(8 ** level)
    block = np.floor(centre / (n0 * dx)).astype(int)
    near = ((block[:, 0] * nb[1] + block[:, 1]) * nb[2] + block[:, 2])
    p = x[near]
    o = block.astype(F) * bext
    i = np.floor((centre - block * n0 * dx) / float(h))
    d = fma(h, i.astype(F) + F(0.5), o) - p
    f = d - half
    c2, f2 = d * d, f * f
    z = d[:, 2]
    xy = c2[:, 0] + c2[:, 1]
    dist = [fma(z, z, xy), (f2[:, 0] + c2[:, 1]) + c2[:, 2], (c2[:, 0] + f2[:, 1]) + c2[:, 2], fma(f[:, 2], f[:, 2], xy)]
    got = [weight, mass[:, 0], mass[:, 1], mass[:, 2]]
    seen = 0
    for q in range(4):
        t = np.maximum(fma(-dist[q], inv, F(1)), F(0))
        w = t * t * t
        # (small weights lose bits to the fixed point: 2^-48 of the largest)
        big = w > 2.0 ** -20
        want = w if q == 0 else w * mp
        assert np.array_equal(got[q][big], want[big]), q
        seen += int(big.sum())
    assert seen > 500


def test_rk3_sum():
    """A constant velocity on each side of a plane, with positions, time step
    and velocities of few bits, so that every sample and stage is exact: k1
    from one side, k2 and k3 from the other."""
    pf = load_pkg()
    lib, msbg = (import_module(pf.__name__ + "." + m) for m in ("_lib", "msbg"))
    print("[gpu] RK3 sum", flush=True)
    h0, nb, n0 = 1.0 / 16, (2, 1, 1), 8
    g = msbg.MSBG(nb, n0=n0, h0=h0, device="cuda:0", max_level=0)
    g.build(np.zeros(2, np.int32))
    right = (g.geometry()[0][:, 0] > 4 * h0)[:, None]
    rng = np.random.default_rng(4)
    n, dt = 512, F(0.75)
    # cells: dt / 2 k1 carries a particle over the plane, 3 dt / 4 k2 too
    x = (rng.integers([16, 56, 56], [32, 72, 72], (n, 3)) / F(16) * F(h0)).astype(F)
    c1, c2, c3 = F(2) / F(9), F(3) / F(9), F(4) / F(9)
    one = torch.zeros(n, dtype=torch.int32, device="cuda")
    prm = lib.MrParams()
    prm.dt = float(dt)
    prm.lo[:], prm.hi[:] = [-10.0] * 3, [10.0] * 3
    other = 0
    for _ in range(16):
        a = np.array([1.0 + rng.integers(0, 16) / 64, *(rng.integers(-3, 4, 2) / 32)], F)
        b = np.array([0.75 + rng.integers(0, 16) / 64, *(rng.integers(-3, 4, 2) / 32)], F)
        fvel = torch.where(right, *(torch.from_numpy(k[None]).cuda() for k in (b, a))).reshape(-1).contiguous()
        end = fma(c1, a, c2 * b)
        want = fma(dt, end + c3 * b, x)
        other += int((want != fma(dt, fma(c3, b, end), x)).sum())
        for nbr in (g.neighbours(), None):
            X, V = torch.from_numpy(x).cuda(), torch.zeros((n, 3), device="cuda")
            ps = lib.MrParticles()
            ps.n, ps.x, ps.v, ps.type, ps.level, ps.defer = n, X.data_ptr(), V.data_ptr(), *([one.data_ptr()] * 3)
            lib.call("pf_mr_advect_near", g.ref(), lib.ptr(nbr), ctypes.byref(ps), ctypes.byref(prm), lib.ptr(fvel),
                     lib.stream())
            assert np.array_equal(X.cpu().numpy(), want)
    assert other > 100  # the case tells the two roundings apart
