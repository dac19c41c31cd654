"""Rounding of Space2's operations along y against the same operations in long double: no larger than that of
a product with the dense operator, whose entries are rounded once from long double, in FP64 (numpy), times
1.5 (the spread of either over a few rows), on rows that fall off as k^-2."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

LD = np.longdouble
CHEB, DIRICHLET, NEUMANN, FOURIER = 0, 1, 2, 4


def _solve(a, b):
    """a x = b by elimination in long double"""
    a, b = a.astype(LD), b.astype(LD)
    n = len(a)
    for k in range(n):
        rows = np.nonzero(a[k + 1:, k])[0] + k + 1
        f = a[rows, k] / a[k, k]
        a[rows, k:] -= f[:, None] * a[k, k:]
        b[rows] -= f[:, None] * b[k]
    x = np.zeros_like(b)
    for k in range(n - 1, -1, -1):
        x[k] = (b[k] - a[k, k + 1:] @ x[k + 1:]) / a[k, k]
    return x


def _operators(kind, n):
    """to_ortho, d/dy and d2/dy2 of it, and from_ortho, in long double (the stencil's own doubles)"""
    i, m = np.arange(n - 2), n - 2
    s = np.zeros((n, m), dtype=LD)
    s[i, i] = 1
    s[i + 2, i] = -1.0 if kind == DIRICHLET else -(i.astype(float) ** 2) / ((i + 2.0) ** 2)
    k, j = np.arange(n)[:, None], np.arange(n)[None, :]
    d = np.where((j > k) & ((j + k) % 2 == 1), 2 * j, 0).astype(LD)
    d[0] /= 2
    return {"ortho": s, "dy": d @ s, "dyy": d @ (d @ s), "proj": _solve(s.T @ s, s.T)}


def _rounding(got, want):
    return float(np.sqrt(((got.astype(LD) - want) ** 2).sum() / (want ** 2).sum()))


@pytest.mark.parametrize("kind", [DIRICHLET, NEUMANN])
@pytest.mark.parametrize("n", [24, 65, 130, 257, 300, 513])
@pytest.mark.parametrize("op", ["ortho", "dy", "dyy", "proj"])
def test_row_operators_round_as_dense_products(n, kind, op):
    from rustpde_amd import Space2
    print("case rounding", n, kind, op, flush=True)
    a, rng = _operators(kind, n)[op], np.random.default_rng(n)
    for k0, n0 in ((FOURIER, 32), (CHEB, 34)):
        sp = Space2((k0, n0), (kind, n))
        shape = sp.shape_ortho if op == "proj" else sp.shape_spectral
        f = rng.standard_normal(shape) / (1.0 + np.arange(shape[0])[:, None] + np.arange(shape[1])) ** 2
        f = f + 0j if sp.is_complex else f
        got = {"ortho": sp.to_ortho, "proj": sp.from_ortho, "dy": lambda v: sp.gradient(v, (0, 1), (1.0, 1.0)),
               "dyy": lambda v: sp.gradient(v, (0, 2), (1.0, 1.0))}[op](f).real
        want, dense = f.real.astype(LD) @ a.T, f.real @ a.astype(float).T
        assert _rounding(got, want) <= 1.5 * _rounding(dense, want), (k0, _rounding(got, want), _rounding(dense, want))


@pytest.mark.parametrize("kind", [DIRICHLET, NEUMANN])
@pytest.mark.parametrize("n", [33, 65, 130, 257, 513])
def test_forward_rounds_as_dense_products(n, kind):
    """Real spaces: dense products along both axes, the one along x as it is (a fast transform along y adds
    its own rounding)."""
    from rustpde_amd import Space2
    print("case forward rounding", n, kind, flush=True)
    m = n - 1
    cosines = np.cos(4 * np.arctan(LD(1)) * np.arange(2 * m).astype(LD) / m)
    t = cosines[(np.arange(n)[:, None] * (m - np.arange(n)[None, :])) % (2 * m)]  # T_k(x_j)
    c = np.ones(n, dtype=LD)
    c[0] = c[-1] = 2
    y = _operators(kind, n)["proj"] @ (LD(2) / m * t / (c[:, None] * c))
    n0 = 24
    mx = n0 - 1
    tx = np.cos(4 * np.arctan(LD(1)) * ((np.arange(n0)[:, None] * (mx - np.arange(n0)[None, :])) % (2 * mx)).astype(LD) / mx)
    cx = np.ones(n0, dtype=LD)
    cx[0] = cx[-1] = 2
    x = LD(2) / mx * tx / (cx[:, None] * cx)
    rng = np.random.default_rng(n)
    g, h = np.linspace(0, 1, n0)[:, None], np.linspace(0, 1, n)[None, :]
    v = sum(np.sin(2 * np.pi * (j + 1) * g + j) * np.sin(np.pi * (j + 1) * h) for j in range(3))
    v = v + 1e-3 * rng.standard_normal(v.shape)
    want, dense = x @ (v.astype(LD) @ y.T), x.astype(float) @ (v @ y.astype(float).T)
    got = Space2((CHEB, n0), (kind, n)).forward(v)
    assert _rounding(got, want) <= 1.5 * _rounding(dense, want), (_rounding(got, want), _rounding(dense, want))
