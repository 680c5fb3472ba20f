"""Level 0 on the half-sweep kernels and on the fused legs: the knobs of either
schedule leave the oracle's bits, and batches whose members' first levels run
in different kernels leave the bits of each member alone."""
import numpy as np
import pytest

from mgpcg_amd import scenes
from oracle import core
from oracle import systems as osys
from test_solve import KNOB_DEFAULTS, _assembled, _x, gpu_solve, set_knobs


def _tile_max(blocks):
    from mgpcg_amd import _lib

    _lib.check(_lib.load().mgpcg_set_option(None, _lib.OPT_TILE_MAX, blocks))


@pytest.fixture(scope="module")
def reference():
    return {}


@pytest.mark.parametrize("tile_max", [0, 768])
@pytest.mark.parametrize("knobs", [
    {}, {"compact": 0}, {"max_grid": 8}, {"max_grid": 64}, {"fuse_p": 1},
    {"restrict_coarse": 0}, {"restrict_coarse": 1}, {"coarse_lds": 0}, {"coarse_max": 0},
    {"compact": 0, "max_grid": 11, "restrict_coarse": 1},
], ids=lambda k: "-".join(f"{a}{b}" for a, b in k.items()) or "defaults")
def test_knobs_on_both_schedules(dev, reference, knobs, tile_max):
    n = 24 if dev == "cpu" else 64
    print(f"case {n}^3 {knobs} tile_max={tile_max} on {dev}", flush=True)
    sysd = scenes.c2_3d(seed=1, n=n, L=3)
    if n not in reference:
        reference[n] = osys.solve(sysd, core.PLAIN, max_iters=6, rel_tol=1e-12)
    set_knobs(**knobs)
    _tile_max(tile_max)
    try:
        x, out, _ = gpu_solve(sysd, dev, "plain", max_iters=6)
    finally:
        set_knobs(**KNOB_DEFAULTS)
        _tile_max(768)
    xr, outr, _ = reference[n]
    assert out["iters"] == outr["iters"]
    assert np.array_equal(x, xr)


@pytest.mark.parametrize("tile_max", [0, 768])
@pytest.mark.parametrize("max_grid", [8, 11, 2048])
def test_batch_of_different_first_levels_equals_alone(dev, tile_max, max_grid):
    """Two members with level 0 on the batched kernels and two, one between them
    and one last, with it in the coarse kernel: finalize finds each member's
    partials in the launch that left them."""
    from mgpcg_amd import batch

    print(f"case tile_max={tile_max} max_grid={max_grid} on {dev}", flush=True)
    mix = [scenes.pool_sphere_system(res, 11 + i, L=3, kind=kind) for i, (res, kind) in enumerate(
        [([24, 20, 28], "pressure"), ([8, 12, 8], "psi"), ([32, 16, 24], "surface"),
         ([8, 8, 16], "volume")])]
    _tile_max(tile_max)
    set_knobs(max_grid=max_grid)
    try:
        solvers = [_assembled(sysd, dev, "mixed") for sysd in mix]
        assert [s.info(0)["coarse_from"] > 0 for s in solvers] == [True, False, True, False]
        res = batch.solve_batch(solvers, max_iters=4, rel_tol=1e-12)
        xs = [_x(s) for s in solvers]
    finally:
        _tile_max(768)
        set_knobs(**KNOB_DEFAULTS)
    for sysd, xb, rb in zip(mix, xs, res):
        xa, ra, _ = gpu_solve(sysd, dev, "mixed", max_iters=4)
        assert ra["iters"] == rb["iters"] and ra["rr"] == rb["rr"]
        assert np.array_equal(xa, xb)


# level 0 in blocks of 256 slots: fewer than the eight groups of a launch, as
# many, a multiple of them and others
@pytest.mark.parametrize("L", [1, 2])
@pytest.mark.parametrize("res,blocks", [([14, 28], 1), ([30, 24], 2), ([62, 50], 7), ([62, 60], 8),
                                        ([62, 66], 9), ([62, 124], 16), ([62, 130], 17),
                                        ([94, 124], 24), ([94, 130], 25)])
def test_dot_products_at_block_counts(dev, res, blocks, L):
    """Finalize sums the partial of every workgroup and no other entry, whatever
    the launch's shape; with two levels the launches of z.r (the legs' blocks of
    24^2) and of the other products leave theirs in different entries."""
    sysd = scenes.pool_sphere_system(res, 9, L=L, kind="pressure")
    slots = (res[0] + 2) * ((res[1] + 3) // 2)
    assert (slots + 255) // 256 == blocks
    set_knobs(coarse_max=0)
    try:
        x, out, _ = gpu_solve(sysd, dev, "plain", max_iters=4)
    finally:
        set_knobs(**KNOB_DEFAULTS)
    xr, outr, _ = osys.solve(sysd, core.PLAIN, max_iters=4, rel_tol=1e-12)
    assert out["iters"] == outr["iters"]
    assert np.array_equal(x, xr)


def test_options_changed_by_another_thread_during_a_solve(dev):
    """The options are process-wide and a solve may run while another thread
    sets them: each iteration keeps those it began with, and the bits are the
    oracle's whatever they are."""
    import threading

    from mgpcg_amd import _lib, mgpcg, systems

    lib = _lib.load()
    sysd = scenes.pool_sphere_system([62, 50], 9, L=2, kind="pressure")
    xr, outr, _ = osys.solve(sysd, core.PLAIN, max_iters=8, rel_tol=1e-12)
    d = systems.upload(sysd, dev)
    set_knobs(coarse_max=0)
    solvers = [mgpcg.MGPCGPoissonSolver(2, sysd["res"], 2, sysd["nu"], sysd["bottom"], device=dev)
               for _ in range(3)]
    stop = threading.Event()
    changes = [0]

    def change():
        rng = np.random.default_rng(1)
        values = [(_lib.OPT_MAX_GRID, (8, 9, 2048)), (_lib.OPT_TILE_MAX, (0, 768)),
                  (_lib.OPT_FUSE_PROLONG, (0, 1)), (_lib.OPT_FUSE_FIRST, (0, 1)),
                  (_lib.OPT_FUSE_P, (0, 1))]
        while not stop.is_set():
            option, of = values[rng.integers(len(values))]
            _lib.check(lib.mgpcg_set_option(None, option, int(of[rng.integers(len(of))])))
            changes[0] += 1

    t = threading.Thread(target=change)
    t.start()
    try:
        for i in range(12):
            s = solvers[i % 3]
            systems.assemble(s, d)
            s.solve(8, rel_tol=1e-12)
            _lib.synchronize(dev)
            assert s.last["iters"] == outr["iters"], (i, changes[0])
            assert np.array_equal(_x(s), xr), (i, changes[0])
    finally:
        stop.set()
        t.join()
        set_knobs(**KNOB_DEFAULTS)
        _tile_max(768)
    assert changes[0] > 10
