"""The coarse kernel with z in LDS and the operators in registers leaves the bits
of its global-memory form, which the oracle checks elsewhere."""
import numpy as np
import pytest
import torch

from mgpcg_amd import scenes
from test_solve import gpu_solve

# all levels in the kernel: one level; the most cells per lane in 3D (2688 per
# colour, all FLUID) and in 2D (3872); two, three and four levels; one cell
# wide; couplings beyond the reciprocal's range
CASES = [([14, 6, 10], 1, "pressure", 1.0), ([16, 14, 24], 2, "psi", 1.0),
         ([88, 88], 3, "psi", 1.0), ([24, 40], 4, "surface", 1.0),
         ([8, 16, 16], 4, "volume", 1.0), ([2, 48, 20], 2, "pressure", 1.0),
         ([32, 48], 3, "pressure", 1e-20), ([8, 16, 12], 2, "pressure", 1e20)]


@pytest.mark.parametrize("res,L,kind,scale", CASES)
def test_lds_coarse_levels_are_the_global_ones(dev, res, L, kind, scale):
    from mgpcg_amd import _lib

    print(f"case {res} L={L} {kind} x{scale:g} on {dev}", flush=True)
    sysd = dict(scenes.pool_sphere_system(res, 3, L=L, kind=kind))
    sysd["scale_A"] *= scale
    lib = _lib.load()
    out = []
    try:
        for lds in (0, 1):
            _lib.check(lib.mgpcg_set_option(None, _lib.OPT_COARSE_LDS, lds))
            out.append(gpu_solve(sysd, dev, "plain", max_iters=5))
    finally:
        _lib.check(lib.mgpcg_set_option(None, _lib.OPT_COARSE_LDS, 1))
    assert out[0][1]["iters"] == out[1][1]["iters"]
    assert np.array_equal(out[0][0], out[1][0])


@pytest.mark.parametrize("p_air", [0.0, 0.01])
@pytest.mark.parametrize("res,L", [([8, 4, 12], 2), ([16, 8, 8], 3), ([16, 32, 16], 5),
                                   ([32, 16, 24], 4), ([32, 48], 4)])
def test_lds_coarse_levels_leave_every_levels_fields(dev, res, L, p_air):
    """After a V-cycle every level's z, on FLUID cells, and r hold what the
    global-memory form leaves."""
    from helpers import random_hierarchy
    from mgpcg_amd import _lib
    from test_kernels import _get, _solver

    print(f"case {res} L={L} p_air={p_air} on {dev}", flush=True)
    h = random_hierarchy(res, L, seed=21, p_fluid=0.97, p_air=p_air)
    r0 = np.random.default_rng(22).standard_normal(res).astype(np.float32)
    lib = _lib.load()
    out = []
    try:
        for lds in (0, 1):
            _lib.check(lib.mgpcg_set_option(None, _lib.OPT_COARSE_LDS, lds))
            s = _solver(h, dev)
            s.debug_set(_lib.FIELD_R, 0, torch.from_numpy(r0))
            s.debug_op(_lib.OP_VCYCLE, 0, 0)
            out.append([_get(s, f, l) for f in (_lib.FIELD_Z, _lib.FIELD_R) for l in range(L)])
    finally:
        _lib.check(lib.mgpcg_set_option(None, _lib.OPT_COARSE_LDS, 1))
    for i, (a, b) in enumerate(zip(*out)):
        cells = (h["gt"][i % L] == 0) | (i >= L)
        assert np.array_equal(a[cells], b[cells]), (("z", "r")[i // L], i % L)
    assert p_air > 0.0 or all((g == 0).any() for g in h["gt"])


@pytest.mark.parametrize("res,L", [([18, 18, 18], 2), ([15, 22, 18], 1), ([89, 88], 1)])
def test_lds_coarse_levels_with_the_most_cells(dev, res, L):
    """The shapes of up to 4096 slots per colour with the most cells, all FLUID:
    2916 and 2970 per colour in 3D, 3916 in 2D."""
    from mgpcg_amd import _lib

    print(f"case {res} L={L} on {dev}", flush=True)
    sysd = scenes.pool_sphere_system(res, 3, L=L, kind="psi")
    lib = _lib.load()
    out = []
    try:
        for lds in (0, 1):
            _lib.check(lib.mgpcg_set_option(None, _lib.OPT_COARSE_LDS, lds))
            out.append(gpu_solve(sysd, dev, "plain", max_iters=3))
    finally:
        _lib.check(lib.mgpcg_set_option(None, _lib.OPT_COARSE_LDS, 1))
    assert out[0][1]["iters"] == out[1][1]["iters"]
    assert np.array_equal(out[0][0], out[1][0])
