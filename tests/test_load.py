"""mgpcg_load leaves what mgpcg_load_level of every level and mgpcg_load_rhs leave."""
import numpy as np
import pytest

from mgpcg_amd import scenes


@pytest.mark.parametrize("res,L,kind,precision", [
    ([16, 8, 24], 3, "pressure", "mixed"), ([6, 10, 2], 1, "psi", "plain"),
    ([8, 40], 4, "surface", "f64"), ([96, 32], 2, "psi", "plain")])
def test_load_is_every_level_and_the_rhs(dev, res, L, kind, precision):
    from mgpcg_amd import _lib, mgpcg, systems

    print(f"case {res} L={L} {kind} {precision} on {dev}", flush=True)
    sysd = scenes.pool_sphere_system(res, 5, L=L, kind=kind)
    d = systems.upload(sysd, dev)
    lib = _lib.load()
    got = []
    for whole in (False, True):
        s = mgpcg.MGPCGPoissonSolver(sysd["dim"], res, L, 2, 10, precision=precision, device=dev)
        systems.assemble(s, d)
        if whole:
            s.load()
        else:
            _lib.check(lib.mgpcg_set_stream(s._h, _lib.stream_handle(s.device)))
            for l in range(L):
                _lib.check(lib.mgpcg_load_level(s._h, l, _lib.ptr(s.grid_type[l]),
                                                _lib.ptr(s.Adiag[l]), _lib.ptr(s.Ax[l])))
            _lib.check(lib.mgpcg_load_rhs(s._h, _lib.ptr(s.b)))
        out = []
        for l in range(L):
            out += [*s.level_flags(l), *s.level_order(l), np.array(s.level_coupling(l))]
        s.load = lambda: None  # solve what was loaded above
        s.solve(4, rel_tol=1e-12)
        _lib.synchronize(dev)
        got.append([o for o in out if o is not None] + [s.x.cpu().numpy()])
    assert len(got[0]) == len(got[1])
    for a, b in zip(*got):
        assert np.array_equal(a, b)
