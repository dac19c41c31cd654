"""The row kernels of Space2 and of the Fourier-axis solves on interleaved complex and on real
arrays, against the oracle, at the edges of their slices (4, 8 and 16 entries per lane and chain:
rows of 512, 1024 and 2048 values; one entry and fewer chains than lanes at the short end), odd
row counts, in place and on arrays that are only 8-byte aligned.

Tolerance 1e-12 of the oracle's largest value, as the other tests of these operations."""
import ctypes

import numpy as np
import pytest

from conftest import rel_err

pytestmark = pytest.mark.gpu

SPACES = [  # (kind0, n0, kind1, n1)
    (4, 8, 1, 6), (4, 8, 2, 7), (4, 16, 0, 33), (4, 8, 1, 131), (4, 8, 2, 512), (4, 8, 1, 513), (4, 8, 0, 1024),
    (4, 8, 1, 1026), (4, 8, 2, 2048), (4, 10, 1, 40), (0, 7, 1, 6), (1, 9, 2, 514), (2, 11, 0, 257), (0, 7, 1, 1025),
]
OPS = ["forward", "backward", "to_ortho", "from_ortho", "gradient"]


def _rand(shape, cplx, seed):
    rng = np.random.default_rng(seed)
    a = rng.standard_normal(shape)
    return a + 1j * rng.standard_normal(shape) if cplx else a


@pytest.mark.parametrize("case", SPACES)
def test_space2_rows_batched(oracle, case):
    from rustpde_amd import Space2
    k0, n0, k1, n1 = case
    print("case rows", case, flush=True)
    sp = Space2((k0, n0), (k1, n1))
    shapes = {"forward": (sp.shape_physical, False), "backward": (sp.shape_spectral, sp.is_complex),
              "to_ortho": (sp.shape_spectral, sp.is_complex), "from_ortho": (sp.shape_ortho, sp.is_complex),
              "gradient": (sp.shape_spectral, sp.is_complex)}
    for op in OPS:
        shp, cplx = shapes[op]
        # coefficients that fall off, as a field's do (a second derivative grows as k^4)
        a = _rand((3,) + shp, cplx, 4) / (1.0 + np.arange(shp[1])) ** 2
        for d in ((1, 0), (2, 0), (0, 1), (0, 2), (1, 1)) if op == "gradient" else (None,):
            got = sp.gradient(a, d, (1.5, 0.75)) if d else getattr(sp, op)(a)
            for b in range(3):
                kw = dict(deriv=d, scale=(1.5, 0.75)) if d else {}
                ref = oracle.space_apply(k0, n0, k1, n1, op, a[b], **kw)
                assert rel_err(got[b], ref) < 1e-12, (op, d, b, rel_err(got[b], ref))


def test_space2_in_place_and_unaligned():
    """to_ortho of a Chebyshev space and a transform in place, and arrays at 8 mod 16 bytes."""
    from rustpde_amd import Space2, _lib
    from rustpde_amd.funspace import _Dev
    L = _lib.load()
    sp = Space2((4, 16), (0, 33))
    v = _rand((2,) + sp.shape_physical, False, 1)
    want = sp.forward(v)
    back = sp.backward(want)
    buf = _Dev(2 * want.nbytes + 16)
    for off in (0, 8):
        at = ctypes.c_void_p(buf.p.value + off)
        far = ctypes.c_void_p(buf.p.value + off + want.nbytes)
        _lib.check(L.rbc_memcpy_h2d(at, want.ctypes.data, want.nbytes))
        _lib.check(L.fs_backward(sp._h, at, far, 2))
        got = np.zeros_like(back)
        _lib.check(L.rbc_memcpy_d2h(got.ctypes.data, far, got.nbytes))
        assert rel_err(got, back) < 1e-14
        one = np.ascontiguousarray(want[0])  # one field, the result over its input
        _lib.check(L.rbc_memcpy_h2d(at, one.ctypes.data, one.nbytes))
        _lib.check(L.fs_backward(sp._h, at, at, 1))
        got0 = np.zeros_like(back[0])
        _lib.check(L.rbc_memcpy_d2h(got0.ctypes.data, at, got0.nbytes))
        assert rel_err(got0, back[0]) < 1e-14
        _lib.check(L.rbc_memcpy_h2d(at, one.ctypes.data, one.nbytes))
        _lib.check(L.fs_gradient(sp._h, at, at, 1, 1, 1.0, 1.0, 1))
        grad = np.zeros_like(one)
        _lib.check(L.rbc_memcpy_d2h(grad.ctypes.data, at, grad.nbytes))
        assert rel_err(grad, sp.gradient(one, (1, 1), (1.0, 1.0))) < 1e-14


@pytest.mark.parametrize("case", [("hholtz", 8, 9, (0.01, 0.02)), ("poisson", 16, 130, (0.25, 1.0)),
                                  ("hholtz", 32, 516, (0.01, 0.02)), ("hholtz", 8, 1027, (1e-3, 1e-3)),
                                  ("hholtz", 10, 40, (0.01, 0.02))])
def test_fourier_solves_batched(oracle, case):
    """Interleaved right-hand sides, and the same over the right-hand sides' own array."""
    from rustpde_amd import Solver, _lib
    from rustpde_amd.funspace import _Dev
    kind, n0, n1, c = case
    print("case fourier solve", case, flush=True)
    g = Solver({"hholtz": 1, "poisson": 2}[kind], (4, n0), (1, n1), c)
    o = oracle.Solver(kind, 4, n0, 1, n1, list(c))
    g.set_tensor(*o.tensor_setup())
    f = _rand((3,) + g.shape_in, True, 3)
    u = g.solve(f)
    for b in range(3):
        assert rel_err(u[b], o.solve(f[b])) < 1e-12, (b, rel_err(u[b], o.solve(f[b])))
    d = _Dev(f.nbytes)
    L = _lib.load()
    _lib.check(L.rbc_memcpy_h2d(d.p, f.ctypes.data, f.nbytes))
    g.solve_device(d.p, d.p, 3)
    got = np.zeros_like(u)
    _lib.check(L.rbc_memcpy_d2h(got.ctypes.data, d.p, got.nbytes))
    assert np.array_equal(got, u)
