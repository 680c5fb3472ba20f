"""The fused V-cycle legs (a level's pre-smoothing with the restriction, and its
prolongation with the post-smoothing, in one launch each) leave the bits of the
half-sweep kernels, which the oracle checks elsewhere."""
import numpy as np
import pytest

from mgpcg_amd import scenes
from test_solve import gpu_solve

# sides around the blocks' 8 (3D) and 24 (2D) cells, remainders of 2 and 4
CASES = [([6, 10, 18], 2, 2, "pressure", "plain"), ([8, 16, 24], 3, 1, "psi", "mixed"),
         ([20, 4, 14], 2, 2, "surface", "plain"), ([12, 28, 20], 3, 2, "volume", "f64"),
         ([24, 48], 2, 2, "pressure", "mixed"), ([50, 22], 2, 1, "psi", "plain"),
         ([28, 100], 3, 2, "surface", "f64")]


@pytest.mark.parametrize("res,L,nu,kind,precision", CASES)
def test_fused_legs_are_the_half_sweeps(dev, res, L, nu, kind, precision):
    from mgpcg_amd import _lib

    print(f"case {res} L={L} nu={nu} {kind} {precision} on {dev}", flush=True)
    sysd = dict(scenes.pool_sphere_system(res, 7, L=L, kind=kind), nu=nu)
    lib = _lib.load()
    out = []
    try:
        for blocks in (0, 768):
            _lib.check(lib.mgpcg_set_option(None, _lib.OPT_TILE_MAX, blocks))
            _lib.check(lib.mgpcg_set_option(None, _lib.OPT_COARSE_MAX_SLOTS, 0))
            out.append(gpu_solve(sysd, dev, precision, max_iters=6))
    finally:
        _lib.check(lib.mgpcg_set_option(None, _lib.OPT_TILE_MAX, 768))
        _lib.check(lib.mgpcg_set_option(None, _lib.OPT_COARSE_MAX_SLOTS, 4096))
    assert out[0][1]["iters"] == out[1][1]["iters"]
    assert np.array_equal(out[0][0], out[1][0])
