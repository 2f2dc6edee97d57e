"""Pressure-solver kernels at the sizes where they can go wrong (edges of
tiles, remainders, smallest and largest of a range), against the FP64
restatement of the V-cycle (oracle/ref_np.py)."""

import numpy as np
import pytest
import torch

from oracle import ref_np as O

pytestmark = pytest.mark.gpu


def _beta(res, rng, walls):
    """Face coefficients over three decades; wall faces closed, or open as a
    caller of MGPCG may leave them (their flux is zero either way)."""
    out = []
    for ax, shape in enumerate(O.face_shapes(res)):
        b = np.exp(rng.uniform(np.log(1e-3), 0.0, size=shape)).astype(np.float32)
        if not walls:
            b[O.wall_mask(shape, ax)] = 0.0
        out.append(b)
    return out


def _vcycle_error(pf, res, precision, walls, pre=3, post=3, min_dim=4, coarsest=60):
    rng = np.random.default_rng(17)
    beta = _beta(res, rng, walls)
    r = rng.standard_normal(res).astype(np.float32)
    r -= r.mean()
    g = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()  # noqa: E731
    solver = pf.MGPCG(res, "cuda:0", pre=pre, post=post, precision=precision, min_dim=min_dim, coarsest=coarsest)
    solver.build_hierarchy(*[g(b) for b in beta])
    z = torch.zeros(res, device="cuda")
    solver.precondition(g(r), z)
    o = O.MGPCGOracle(res, pre=pre, post=post, min_dim=min_dim, coarsest=coarsest)
    o.build_hierarchy(*beta)
    ref = o.precondition(r.astype(np.float64))
    return float(np.linalg.norm(z.cpu().numpy() - ref) / np.linalg.norm(ref))


# coarsest levels of 3 to 8 pairs of cells per thread (from 6 on the z faces
# are in LDS), odd and even extents along k, then one too large for the kernel
@pytest.mark.parametrize("coarsest", [(27, 19, 13), (31, 23, 9), (33, 25, 11), (27, 27, 15), (29, 27, 17),
                                      (25, 25, 25), (31, 33, 8), (41, 37, 12), (35, 33, 21)])
@pytest.mark.parametrize("walls", [False, True])
def test_coarsest_level_in_one_workgroup(pf, coarsest, walls):
    """The coarsest level's 60 sweeps and mean removal where it is too large
    for the LDS V-cycle.  FP32 against FP64 over a V-cycle: the bound of the
    V-cycle tests in test_gpu_parity.py."""
    res = tuple(2 * n for n in coarsest)
    print(f"[gpu] coarsest {coarsest} walls={walls}", flush=True)
    assert _vcycle_error(pf, res, "fp32", walls) < 2e-5


@pytest.mark.parametrize("precision,bound", [("bf16", 2e-2), ("fp16", 3e-3)])
def test_coarsest_level_in_one_workgroup_16_bit(pf, precision, bound):
    """16-bit V-cycles: the level above stores its iterate once per colour of
    its 3 + 3 sweeps, 12 relative roundings of 2^-9 or 2^-12 (2.3e-2, 2.9e-3)."""
    print(f"[gpu] coarsest 16-bit {precision}", flush=True)
    assert _vcycle_error(pf, (54, 38, 26), precision, False) < bound


# one workgroup from the largest level it takes down: register levels only,
# LDS levels below them (min_dim 1), one register level, a coarsest level by
# its sweeps (729 cells), by its matrix alone, and a whole grid by its sweeps
@pytest.mark.parametrize("res,min_dim", [((16, 16, 16), 4), ((32, 32, 32), 1), ((16, 16, 16), 1), ((64, 8, 8), 2),
                                         ((24, 12, 20), 4), ((18, 18, 18), 4), ((7, 8, 9), 4), ((11, 13, 9), 4),
                                         ((128, 16, 8), 4)])
@pytest.mark.parametrize("walls", [False, True])
@pytest.mark.parametrize("pre,post", [(3, 3), (1, 2)])
def test_small_hierarchy_in_one_workgroup(pf, res, min_dim, walls, pre, post):
    """FP32 against FP64 over a V-cycle, the bound of the tests above."""
    print(f"[gpu] small hierarchy {res} min_dim={min_dim} walls={walls} {pre}+{post}", flush=True)
    assert _vcycle_error(pf, res, "fp32", walls, pre, post, min_dim) < 2e-5


# 8 x 8 x 32 tiles: whole, cut along every axis, 1152 of them; 8 x 8 x 64 tiles
# beside them; 8 x 8 x 16 where the longer ones would be padded most
@pytest.mark.parametrize("res,precision", [((96, 88, 96), "fp32"), ((100, 90, 84), "fp32"), ((104, 120, 100), "bf16"),
                                           ((192, 128, 96), "fp16"), ((128, 64, 192), "bf16"),
                                           ((260, 256, 12), "fp32"), ((260, 256, 16), "bf16"),
                                           ((148, 140, 36), "bf16"), ((212, 208, 48), "fp32")])
def test_sweep_tiles_equal_half_sweeps(pf, res, precision):
    """The fused sweeps of every tile shape against two half-sweep launches
    per sweep, bit for bit, over a V-cycle and a solve of 6 iterations (the
    inner products in a kernel of their own in both)."""
    print(f"[gpu] sweep tiles {res} {precision}", flush=True)
    rng = np.random.default_rng(3)
    g = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()  # noqa: E731
    beta = [g(b) for b in _beta(res, rng, False)]
    r = g(rng.standard_normal(res).astype(np.float32))
    out = []
    for fused in (True, False):
        s = pf.MGPCG(res, "cuda:0", pre=2, post=2, precision=precision, fused_smoother=fused, fold_dots=False)
        s.build_hierarchy(*beta)
        z, p = torch.zeros_like(r), torch.zeros_like(r)
        s.precondition(r, z)
        it, rel = s.solve(r, p, tol=1e-30, max_iter=6)
        out.append((z.cpu().numpy(), p.cpu().numpy(), it, rel))
    assert np.array_equal(out[0][0], out[1][0]) and np.array_equal(out[0][1], out[1][1])
    assert out[0][2:] == out[1][2:]


def _solve_both(pf, res, precision, tell, pre=3, post=3, **kw):
    """Six FPCG iterations and a V-cycle with two settings of a solver."""
    rng = np.random.default_rng(21)
    g = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()  # noqa: E731
    beta = [g(b) for b in _beta(res, rng, False)]
    r = g(rng.standard_normal(res).astype(np.float32))
    out = []
    for v in (True, False):
        s = pf.MGPCG(res, "cuda:0", pre=pre, post=post, precision=precision, **{tell: v}, **kw)
        s.build_hierarchy(*beta)
        z, p = torch.zeros_like(r), torch.zeros_like(r)
        s.precondition(r, z)
        it, rel = s.solve(r, p, tol=1e-30, max_iter=6)
        out.append((z.cpu().numpy(), p.cpu().numpy().astype(np.float64), it, rel))
    return out


# one partial per tile: 1152 and cut 8 x 8 x 32 tiles, 8 x 8 x 16 and 4 x 8 x 16
# (whole and cut), cut 8 x 8 x 64 ones, and the post phase of a level 0 with cut
# tiles
@pytest.mark.parametrize("res,split", [((192, 128, 96), False), ((100, 90, 84), False), ((80, 80, 80), False),
                                       ((64, 64, 64), True), ((52, 60, 44), True), ((32, 32, 32), True),
                                       ((40, 48, 56), True),
                                       ((124, 100, 128), False), ((40, 48, 56), False), ((22, 30, 26), False)])
@pytest.mark.parametrize("precision", ["fp32", "bf16", "fp16"])
def test_inner_products_of_every_tile_shape(pf, res, split, precision):
    """The CG's inner products from the last level-0 kernel of a V-cycle
    against a kernel of their own.  The two differ by the order of FP64
    additions, so a scalar that scales a vector differs by one unit in the
    last place of FP32 at most, and rarely; six iterations carry 1e-5 of the
    result, as in the solver tests."""
    print(f"[gpu] inner products {res} split={split} {precision}", flush=True)
    a, b = _solve_both(pf, res, precision, "fold_dots", split_levels=split)
    assert np.array_equal(a[0], b[0]) and a[2] == b[2] == 6
    assert np.abs(a[1] - b[1]).max() < 1e-5 * np.abs(b[1]).max()


# tiles of 8 x 8 x 16 cells cut along k and along every axis, of 4 x 4 x 8 cut
# along every axis and along k, on level 0 and on the levels below
@pytest.mark.parametrize("res", [(40, 48, 56), (36, 28, 44), (22, 30, 26), (20, 28, 12), (60, 68, 76)])
@pytest.mark.parametrize("pre,post", [(3, 3), (1, 2), (2, 1)])
@pytest.mark.parametrize("precision", ["fp32", "bf16", "fp16"])
def test_phases_with_cut_tiles_equal_sweeps(pf, res, pre, post, precision):
    """Smoothing phases in one launch each against one launch per sweep, bit
    for bit, over a V-cycle and a solve (which takes its residual test from
    level 0's first kernel)."""
    print(f"[gpu] phases {res} {pre}+{post} {precision}", flush=True)
    a, b = _solve_both(pf, res, precision, "split_levels", pre, post, fold_dots=False)
    assert np.array_equal(a[0], b[0]) and np.array_equal(a[1], b[1]) and a[2:] == b[2:]


def _residual(beta, b, p):
    """max |b - mean b - A p| / max |b - mean b| in FP64."""
    b, p = b.double(), p.double()
    b = b - b.mean()
    r = b.clone()
    for a, f in enumerate(beta):
        n = p.shape[a]
        flux = f.double().narrow(a, 1, n - 1) * (p.narrow(a, 1, n - 1) - p.narrow(a, 0, n - 1))
        r.narrow(a, 0, n - 1).add_(flux)
        r.narrow(a, 1, n - 1).sub_(flux)
    return float(r.abs().max() / b.abs().max())


# nx odd, one axis too short, more than 1024 sweep tiles; nz even throughout,
# so that level 0 has fused sweeps
@pytest.mark.parametrize("res", [(25, 24, 32), (6, 64, 64), (161, 160, 160)])
@pytest.mark.parametrize("precision", ["fp32", "bf16", "fp16"])
def test_solve_on_a_grid_that_cannot_be_halved(pf, res, precision):
    """A hierarchy of one level above the sizes that one workgroup takes.  The
    FP32 recursive residual follows b - A p to within the rounding of its
    updates, some 1e-6 of max |b| here."""
    print(f"[gpu] one level {res} {precision}", flush=True)
    rng = np.random.default_rng(8)
    g = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()  # noqa: E731
    beta = [g(b) for b in _beta(res, rng, False)]
    b = g(rng.standard_normal(res).astype(np.float32))
    s = pf.MGPCG(res, "cuda:0", pre=3, post=3, precision=precision)
    assert s.nlev == 1 and s.small_from == 1
    s.build_hierarchy(*beta)
    p = torch.zeros_like(b)
    for _ in range(2):  # the second from the captured graphs
        it, rel = s.solve(b, p, tol=1e-4, max_iter=400)
        assert 0 < it < 400 and rel < 1e-4
        assert _residual(beta, b, p) < 1.2e-4


@pytest.mark.parametrize("res", [(25, 24, 32), (25, 24, 31), (50, 48, 62)])
@pytest.mark.parametrize("coarsest", [1, 7, 8])
def test_odd_number_of_coarsest_sweeps(pf, res, coarsest):
    """An odd number of fused sweeps ends in the level's second buffer: the
    result of a one-level hierarchy is moved from there (nz even; in place for
    an odd nz; and on a level below another)."""
    print(f"[gpu] coarsest sweeps {res} {coarsest}", flush=True)
    assert _vcycle_error(pf, res, "fp32", False, coarsest=coarsest) < 2e-5
