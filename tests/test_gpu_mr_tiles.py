"""The tiled adaptive P2G against the per-particle kernel, bit for bit: every
class of particle (own level, one level coarser, two coarser, finer, across
2:1 jumps, outside the grid) on blocks of one cell per axis up to several
tiles per block."""

import numpy as np
import pytest

from conftest import load_pkg

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nb,n0,max_level,seed", [
    ((3, 2, 2), 16, 2, 1),   # 16^3, 8^3 and 4^3 cells per block: 8 tiles, 1 tile, part of a tile
    ((2, 3, 2), 32, 1, 2),   # 64 and 8 tiles per block
    ((4, 3, 5), 8, 3, 3),    # down to one cell per block
    ((5, 4, 3), 2, 1, 4),    # blocks of 2 and of 1 cells: every support crosses blocks
    ((1, 1, 1), 8, 0, 5),    # one block: every neighbour is missing
    ((2, 2, 1), 64, 6, 6),   # 512 tiles down to one cell per block
    ((3, 2, 2), 64, 1, 7),
])
def test_tiled_p2g_equals_per_particle_atomics(nb, n0, max_level, seed):
    from importlib import import_module
    pf = load_pkg()
    cfgm, mrs = (import_module(pf.__name__ + "." + m) for m in ("config", "mr_sim"))
    print(f"[gpu] tiled adaptive P2G {nb} n0={n0} max_level={max_level}", flush=True)
    rng = np.random.default_rng(seed)
    dx = 0.37 / n0  # no power of two: cell centres round
    cfg = cfgm.Config(res=tuple(n * n0 for n in nb), dx=dx, ppc=27, droplets=False)
    levels = rng.integers(0, max_level + 1, size=int(np.prod(nb)))
    sim = mrs.AdaptiveSimulator(cfg, nb, n0=n0, max_level=max_level, frozen_levels=levels)
    L = np.array(nb) * n0 * dx
    n = 150000  # (fewer than 2^17 are all walked)
    x = rng.random((n, 3)) * L
    x[: n // 50] = rng.random((n // 50, 3)) * (1.2 * L) - 0.1 * L       # some outside the box
    on = rng.integers(0, n, size=n // 20)
    x[on] = np.round(x[on] / dx) * dx                                   # on faces and corners
    lev = rng.integers(0, max_level + 1, size=n).astype(np.int32)
    sim.set_particles(x.astype(np.float32), rng.standard_normal((n, 3)).astype(np.float32),
                      rng.integers(0, 2, size=n).astype(np.int32), lev)
    sim._rebuild_grid(1e-3)
    prm = sim._params(1e-3, sim._max_speed())
    out = []
    for sorted_ in (True, False, True):  # the second tiled run: on a used scratch buffer
        sim.p2g_sorted = sorted_
        sim.stage_p2g(prm)
        out.append({k: getattr(sim, k).cpu().numpy().copy() for k in ("cwsum", "phi", "fmass", "fvel", "is_liquid")})
    for k in out[0]:
        assert np.array_equal(out[0][k], out[1][k]), k
        assert np.array_equal(out[2][k], out[1][k]), k
    assert np.abs(out[0]["fmass"]).max() > 0


@pytest.mark.parametrize("n", [1, 1000, 131071, 131072, 400000])
@pytest.mark.parametrize("levels,plev", [("checker", 0), ("checker", 1), ("small", 2), ("one", 0)])
def test_tiled_p2g_leaves_particles_to_the_walk(n, levels, plev):
    """Few particles (all walked), tiles that leave more than 512 particles to
    the walk (all blocks facing others of another level, and particles finer
    than their block), blocks of 4, 2 and 1 cells per axis among larger ones."""
    from importlib import import_module
    pf = load_pkg()
    cfgm, mrs = (import_module(pf.__name__ + "." + m) for m in ("config", "mr_sim"))
    print(f"[gpu] tiled adaptive P2G, walk {n} {levels} {plev}", flush=True)
    rng = np.random.default_rng(n)
    nb, n0, dx = (5, 4, 7), 8, 0.37 / 8
    if levels == "checker":
        n0 = 16
    lv = {"checker": np.indices(nb).sum(0).ravel() % 2, "small": rng.integers(1, 4, 140), "one": np.zeros(140)}[levels]
    cfg = cfgm.Config(res=tuple(k * n0 for k in nb), dx=dx, ppc=27, droplets=False)
    sim = mrs.AdaptiveSimulator(cfg, nb, n0=n0, max_level=3, frozen_levels=lv.astype(int))
    x = (rng.random((n, 3)) * np.array(nb) * n0 * dx).astype(np.float32)
    x[::101] *= 1.3  # some outside
    sim.set_particles(x, rng.standard_normal((n, 3)).astype(np.float32), rng.integers(0, 2, n).astype(np.int32),
                      np.full(n, plev, np.int32))
    sim._rebuild_grid(1e-3)
    prm = sim._params(1e-3, sim._max_speed())
    out = []
    for sorted_ in (True, False, True):
        sim.p2g_sorted = sorted_
        sim.stage_p2g(prm)
        out.append({k: getattr(sim, k).cpu().numpy().copy() for k in ("cwsum", "phi", "fmass", "fvel", "is_liquid")})
    for k in out[0]:
        assert np.array_equal(out[0][k], out[1][k]) and np.array_equal(out[2][k], out[1][k]), k


def test_tiled_p2g_on_coarse_levels_of_large_blocks():
    """8192 blocks of 512^3 finest cells, all at one cell per block: as many
    tiles as blocks, where 2^31 would be one for every 8^3 finest cells."""
    from importlib import import_module
    pf = load_pkg()
    cfgm, mrs = (import_module(pf.__name__ + "." + m) for m in ("config", "mr_sim"))
    print("[gpu] tiled adaptive P2G, one cell per 512^3 block", flush=True)
    rng = np.random.default_rng(8)
    nb, n0, dx = (32, 16, 16), 512, 0.37 / 512
    cfg = cfgm.Config(res=tuple(n * n0 for n in nb), dx=dx, ppc=27, droplets=False)
    sim = mrs.AdaptiveSimulator(cfg, nb, n0=n0, max_level=9, frozen_levels=np.full(int(np.prod(nb)), 9))
    n = 150000
    x = (rng.random((n, 3)) * np.array(nb) * n0 * dx).astype(np.float32)
    sim.set_particles(x, rng.standard_normal((n, 3)).astype(np.float32), np.ones(n, np.int32),
                      rng.choice([8, 9], n).astype(np.int32))
    sim._rebuild_grid(1e-3)
    prm = sim._params(1e-3, sim._max_speed())
    out = []
    for sorted_ in (True, False):
        sim.p2g_sorted = sorted_
        sim.stage_p2g(prm)
        out.append({k: getattr(sim, k).cpu().numpy().copy() for k in ("cwsum", "phi", "fmass", "fvel", "is_liquid")})
    for k in out[0]:
        assert np.array_equal(out[0][k], out[1][k]), k
    assert np.abs(out[0]["fmass"]).max() > 0


@pytest.mark.parametrize("n0,level", [(16, 0), (32, 1), (8, 0)])
@pytest.mark.parametrize("coarser", [0, 1])
def test_particles_at_tile_edges_are_splatted_once(n0, level, coarser):
    """Particles of the tiles' level and one level coarser, on tile and block
    edges and a few units in the last place beside them, with a spacing that
    is no power of two: the two tile kernels and the walk share them out
    without losing one or taking one twice."""
    from importlib import import_module
    pf = load_pkg()
    cfgm, mrs = (import_module(pf.__name__ + "." + m) for m in ("config", "mr_sim"))
    print(f"[gpu] tile edges n0={n0} level={level} coarser={coarser}", flush=True)
    rng = np.random.default_rng(6)
    nb, dx = (5, 4, 3), 0.37 / 11
    cfg = cfgm.Config(res=tuple(n * n0 for n in nb), dx=dx, ppc=27, droplets=False)
    sim = mrs.AdaptiveSimulator(cfg, nb, n0=n0, max_level=2, frozen_levels=np.full(int(np.prod(nb)), level))
    n, edge = 150000, (8 << level) * np.float32(dx)
    cells = np.array(nb) * n0 // (8 << level)
    x = (rng.random((n, 3)) * np.array(nb) * n0 * dx).astype(np.float32)
    on = rng.integers(0, 3, n)  # the axis along which it sits at an edge
    at = (rng.integers(1, np.maximum(cells, 2)[on], n).astype(np.float32) * edge).view(np.int32)
    x[np.arange(n), on] = (at + rng.integers(-3, 4, n).astype(np.int32)).view(np.float32)
    lev = np.full(n, level + coarser, np.int32)
    sim.set_particles(x, rng.standard_normal((n, 3)).astype(np.float32), np.ones(n, np.int32), lev)
    sim._rebuild_grid(1e-3)
    prm = sim._params(1e-3, sim._max_speed())
    out = []
    for sorted_ in (True, False):
        sim.p2g_sorted = sorted_
        sim.stage_p2g(prm)
        out.append({k: getattr(sim, k).cpu().numpy().copy() for k in ("cwsum", "phi", "fmass", "fvel", "is_liquid")})
    for k in out[0]:
        assert np.array_equal(out[0][k], out[1][k]), k


@pytest.mark.parametrize("nb,n0,levels", [((8, 8, 8), 2, "one"), ((3, 3, 3), 4, "jump"), ((1, 2, 1), 4, "one"),
                                          ((7, 7, 9), 2, "one")])
def test_coarse_level_matrix_matches_the_sweeps(nb, n0, levels):
    """The coarsest level's matrix (rows of 6 couplings, and of up to 24 next
    to a 2:1 jump; 8 to 512 cells, whole and partial workgroups of its
    product) against the launched sweeps in FP32: 80 sweeps of FP32 rounding,
    held to 2e-4 of the solution's size as in the V-cycle tests."""
    from importlib import import_module
    import torch
    pf = load_pkg()
    lib, msbg, mgm = (import_module(pf.__name__ + "." + m) for m in ("_lib", "msbg", "mr_multigrid"))
    print(f"[gpu] coarse matrix {nb} n0={n0} {levels}", flush=True)
    rng = np.random.default_rng(4)
    top = {2: 1, 4: 2}[n0]
    lv = np.full(int(np.prod(nb)), top, np.int32)
    if levels == "jump":
        lv[len(lv) // 2] = top - 1
    g = msbg.MSBG(nb, n0=n0, h0=0.1, device="cuda:0", max_level=top)
    g.build(lv)
    assert g.ncells <= 512
    mg = mgm.MRMultigrid(g, min_cells=10 ** 9)
    bface = torch.from_numpy((0.1 + rng.random(3 * g.ncells)).astype(np.float32)).cuda()
    mg.build_hierarchy(bface)
    c = mg.levels[-1]
    b = torch.from_numpy(rng.standard_normal(c.n).astype(np.float32)).cuda()
    c.b.copy_(b - b.mean())
    assert mg.coarsest_mode == "matrix"
    got = torch.zeros_like(c.p)
    lib.call("pf_msbg_coarse_apply", lib.ptr(mg._coarse_op), lib.ptr(c.b), lib.ptr(got), c.n, lib.stream())
    c.p.zero_()
    mg._smooth(c, mg.coarsest_sweeps)
    ref = (c.p - c.p.double().mean().float()).double()
    assert float((got.double() - ref).abs().max()) < 2e-4 * float(ref.abs().max())
