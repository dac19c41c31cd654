"""Fields of one call do not touch each other: with an infinity in one of them, or values 1e12 as large, the
others are those of a call of their own, bit for bit.  Odd numbers of rows along x (a transform along y takes
two rows at a time), even ones, and Fourier axes; all of Space2's operations and the batched solves."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

CHEB, DIRICHLET, NEUMANN, FOURIER = 0, 1, 2, 4


def _rand(shape, cplx, seed):
    rng = np.random.default_rng(seed)
    k = 1.0 + np.arange(shape[-2])[:, None] + np.arange(shape[-1])
    a = rng.standard_normal(shape) / k ** 2
    return a + 1j * rng.standard_normal(shape) / k ** 2 if cplx else a


def _check(call, a):
    for spoil in (np.inf, 1e12):
        b = a.copy()
        b[1] = b[1] * 1e12 if spoil == 1e12 else b[1]
        if spoil != 1e12:
            b[1, :, 0] = spoil
        got = call(b)
        for i in (0, 2):
            assert np.array_equal(got[i], call(a[i])), (spoil, i)


@pytest.mark.parametrize("case", [(CHEB, 7, CHEB, 33), (NEUMANN, 33, NEUMANN, 129), (DIRICHLET, 9, DIRICHLET, 65),
                                  (DIRICHLET, 35, NEUMANN, 40), (CHEB, 8, NEUMANN, 33), (FOURIER, 16, NEUMANN, 65),
                                  (FOURIER, 10, DIRICHLET, 33), (FOURIER, 12, CHEB, 21)])
def test_fields_of_a_space(case):
    from rustpde_amd import Space2
    k0, n0, k1, n1 = case
    print("case fields", case, flush=True)
    sp = Space2((k0, n0), (k1, n1))
    c = sp.is_complex
    for name, shape, cplx in (("forward", sp.shape_physical, False), ("backward", sp.shape_spectral, c),
                              ("to_ortho", sp.shape_spectral, c), ("from_ortho", sp.shape_ortho, c)):
        _check(getattr(sp, name), _rand((3,) + tuple(shape), cplx, 1))
    for d in ((1, 0), (0, 1), (0, 2), (1, 1)):
        _check(lambda v: sp.gradient(v, d, (1.5, 0.75)), _rand((3,) + tuple(sp.shape_spectral), c, 2))


@pytest.mark.parametrize("case", [(0, DIRICHLET, 33, NEUMANN, 35), (1, NEUMANN, 35, DIRICHLET, 33),
                                  (2, FOURIER, 16, NEUMANN, 33), (1, FOURIER, 10, DIRICHLET, 40)])
def test_fields_of_a_solve(case):
    from rustpde_amd import Solver
    kind, k0, n0, k1, n1 = case
    print("case fields of a solve", case, flush=True)
    s = Solver(kind, (k0, n0), (k1, n1), (0.25, 1.0) if kind == 2 else (0.01, 0.02))
    _check(s.solve, _rand((5,) + tuple(s.shape_in), s.is_complex, 3))
