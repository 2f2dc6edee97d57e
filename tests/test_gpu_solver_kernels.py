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


def _vcycle_error(pf, res, precision, walls, pre=3, post=3):
    rng = np.random.default_rng(17)
    beta = _beta(res, rng, walls)
    r = rng.standard_normal(res).astype(np.float32)
    r -= r.mean()
    g = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()  # noqa: E731
    solver = pf.MGPCG(res, "cuda:0", pre=pre, post=post, precision=precision)
    solver.build_hierarchy(*[g(b) for b in beta])
    z = torch.zeros(res, device="cuda")
    solver.precondition(g(r), z)
    o = O.MGPCGOracle(res, pre=pre, post=post)
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
    """16-bit V-cycles: the bound is 8 units of the storage format's relative
    rounding (2^-9, 2^-12), one per smoothing pass of the level above."""
    print(f"[gpu] coarsest 16-bit {precision}", flush=True)
    assert _vcycle_error(pf, (54, 38, 26), precision, False) < bound
