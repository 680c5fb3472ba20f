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


# the FP32 limit is 768 blocks in 3D, the FP64 one 512, the 2D one 3072
@pytest.mark.parametrize("res,nu,precision,limit,legs", [
    ([16, 16, 16], 2, "plain", 8, True), ([16, 16, 16], 2, "plain", 7, False),
    ([16, 16, 16], 1, "plain", 768, False), ([16, 16, 16], 1, "f64", 768, False),
    ([16, 24, 16], 2, "f64", 18, True), ([16, 24, 16], 2, "f64", 17, False),
    ([48, 48], 2, "plain", 1, True), ([48, 72], 2, "f64", 1, False),
    ([48, 48], 1, "mixed", 1, True), ([48, 48], 1, "f64", 1, True)])
def test_where_the_fused_legs_run(dev, res, nu, precision, limit, legs):
    """The rule on blocks, smoothing steps and type, by the launches of a solve."""
    from mgpcg_amd import _lib

    lib = _lib.load()
    if not hasattr(lib, "hipemu_launches"):
        pytest.skip("counts the emulator's launches")
    sysd = dict(scenes.pool_sphere_system(res, 7, L=2, kind="psi"), nu=nu)
    count = []
    try:
        _lib.check(lib.mgpcg_set_option(None, _lib.OPT_COARSE_MAX_SLOTS, 0))
        for blocks in (0, limit):
            _lib.check(lib.mgpcg_set_option(None, _lib.OPT_TILE_MAX, blocks))
            n = lib.hipemu_launches()
            gpu_solve(sysd, dev, precision, max_iters=1)
            count.append(lib.hipemu_launches() - n)
    finally:
        _lib.check(lib.mgpcg_set_option(None, _lib.OPT_TILE_MAX, 768))
        _lib.check(lib.mgpcg_set_option(None, _lib.OPT_COARSE_MAX_SLOTS, 4096))
    assert (count[1] < count[0]) == legs and (count[1] == count[0]) != legs
