"""The tiled transpose of G2P + RK3 against the per-particle one: partial
tiles, both phases in a tile, particles outside the bins, solids, stages that
leave the staged box, and each flag on its own."""

import ctypes

import numpy as np
import pytest
import torch

from conftest import load_pkg

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def pf():
    return load_pkg()


def _sim(pf, res, ppc, solids, states, seed=3):
    cfg = pf.Config(res=res, dx=1.0 / max(res), ppc=ppc, droplets=False, gravity=(0.0, 0.0, -9.81), seed=seed)
    pos, vel, pt = pf.scenes.dam_break(cfg, frac=(0.45, 1.0, 0.6))
    rng = np.random.default_rng(seed)
    vel = vel + rng.standard_normal(vel.shape).astype(np.float32)
    sim = pf.Simulator(cfg)
    sim.set_particles(pos, vel, pt)
    if solids:
        m = np.zeros(res, bool)
        m[res[0] // 2:res[0] // 2 + 2, :, : res[2] // 2] = True
        sim.set_solids(m)
    if states:  # droplets and dead particles, outside the bins
        st = rng.choice([0, 0, 0, 1, 2], size=len(pos)).astype(np.int32)
        sim.pstate.copy_(torch.from_numpy(st))
    for f in (sim.vel, sim.dvel, sim.vel_liq):
        for a in range(3):
            f[a].copy_(torch.from_numpy(rng.standard_normal(tuple(f[a].shape)).astype(np.float32)))
    return cfg, sim


def _run(pf, sim, flags, dt, binned, gx, gv):
    L = pf.sim._lib
    fs = sim.face_shapes
    grids = [[torch.zeros(s, device="cuda") for s in fs] for _ in range(3)]
    out = [torch.empty_like(gx), torch.empty_like(gv)]
    a = sim._g2p_args(flags, dt)
    bins = [L.ptr(sim.perm), L.ptr(sim.cell_start), L.ptr(sim._n_active)] if binned else []
    L.call("pf_adj_g2p_advect_binned" if binned else "pf_adj_g2p_advect", ctypes.byref(a), *bins, L.ptr(gx),
           L.ptr(gv), L.ptr(out[0]), L.ptr(out[1]), *[L.ptr3(g) for g in grids], L.stream())
    torch.cuda.synchronize()
    return out, grids


@pytest.mark.parametrize("res,ppc,solids,states,cfl,parts", [
    ((16, 16, 16), 8, False, False, 0.9, 7),
    ((13, 9, 21), 8, False, True, 0.9, 7),
    ((24, 16, 11), 27, True, True, 0.9, 7),
    ((17, 8, 10), 8, False, False, 3.0, 7),   # stages leave the staged box
    ((9, 12, 16), 8, False, False, 0.9, 1),   # G2P only
    ((9, 12, 16), 8, True, False, 0.9, 6),    # advection and walls only
])
def test_tiled_adjoint_equals_per_particle(pf, res, ppc, solids, states, cfl, parts):
    print(f"[gpu] tiled adjoint {res} ppc={ppc} solids={solids} states={states} cfl={cfl}", flush=True)
    cfg, sim = _sim(pf, res, ppc, solids, states)
    L = pf.sim._lib
    sim._bin()
    flags = (L.GA_G2P if parts & 1 else 0) | (L.GA_ADVECT if parts & 2 else 0) | (L.GA_REFLECT if parts & 4 else 0)
    dt = cfl * cfg.dx / 3.0  # fields are N(0, 1)
    g = torch.Generator(device="cuda").manual_seed(1)
    gx, gv = (torch.randn(sim.px.shape, generator=g, device="cuda") for _ in range(2))
    (x0, v0), f0 = _run(pf, sim, flags, dt, False, gx, gv)
    (x1, v1), f1 = _run(pf, sim, flags, dt, True, gx, gv)

    def close(a, b):
        # FP32 sums of up to a few hundred terms, and gradients by differences
        # instead of weighted sums: 2^-24 x ~100 of the field's norm.  A
        # particle whose floor(x / dx) differs between x / dx and x * (1 / dx)
        # sits on a kink of the trilinear sample, where both one-sided
        # gradients are valid: such rows (at most a few) are left out.
        a, b = a.double().reshape(-1), b.double().reshape(-1)
        scale = b.norm() / max(b.numel(), 1) ** 0.5
        bad = (a - b).abs() > 1e-3 * torch.maximum(scale, b.abs())
        assert bad.float().mean() < 1e-4
        assert float(((a - b)[~bad]).norm()) <= 1e-5 * float(b.norm()) + 1e-30

    close(x1, x0)
    close(v1, v0)
    for k in range(3):
        for a in range(3):
            close(f1[k][a], f0[k][a])
