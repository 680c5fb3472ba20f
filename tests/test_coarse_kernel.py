"""The coarse kernel with z in LDS and the operators in registers leaves the bits
of its global-memory form, which the oracle checks elsewhere."""
import numpy as np
import pytest

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
