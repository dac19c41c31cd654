"""Batches large enough for the variants that small ones do not reach: the 64 x 64 tiles of the parity-class
products (a wavefront per tile, its own order of accumulation), for every operator kind and both store
orders, and row solves of eight entries a lane with four right-hand sides a wavefront.  The size rules are
restated here, so that a case that no longer selects its variant fails.

The same call on one field takes small tiles and single rows; the sums are formed in one order everywhere, so
its results have the same bits.  One entry is also compared with the oracle, to the 1e-12 of other tests of
these operations (1e-9 across two eigen-decompositions)."""
import numpy as np
import pytest

from conftest import rel_err

pytestmark = pytest.mark.gpu

CHEB, DIRICHLET, NEUMANN = 0, 1, 2


def _groups(k):
    q = (k + 31) // 32
    if q <= 4:
        return 4 * q
    up = lambda c: (q + c - 1) // c * c  # noqa: E731
    best = 4
    for c in (3, 2):
        if up(c) < up(best):
            best = c
    return 4 * up(best)


def _large(products):
    """products of one launch: (rows, inputs of the longer class, classes, columns, entries)"""
    size = size64 = 0
    for m, k, classes, n, entries in products:
        per = classes * entries * _groups(k)
        size += -(-n // 16) * -(-m // 16) * per
        size64 += 16 * -(-n // 64) * -(-m // 64) * per
    return size >= 400000 and 10 * size64 <= 11 * size


def _rand(shape, seed):
    rng = np.random.default_rng(seed)
    k = np.arange(shape[-2])[:, None] + np.arange(shape[-1])[None, :]
    return rng.standard_normal(shape) / (1.0 + k) ** 2


def _same_bits(call, a, got):
    for b in (0, 1, len(a) // 2, len(a) - 1):
        assert np.array_equal(got[b], call(a[b])), b


def test_solve_of_blocks_and_undivided(oracle):
    from rustpde_amd import Solver
    n0, n1, batch = 258, 190, 136
    print("case large batch hholtz", n0, n1, batch, flush=True)
    assert _large([(128, 129, 2, n1, batch)]) and _large([(128, 128, 2, n1 - 2, batch)])
    assert _large([(256, 258, 1, n1, batch)]) and _large([(256, 256, 1, n1 - 2, batch)])
    s = Solver(1, (DIRICHLET, n0), (DIRICHLET, n1), (0.01, 0.02))
    o = oracle.Solver("hholtz", DIRICHLET, n0, DIRICHLET, n1, [0.01, 0.02])
    f = _rand((batch, n0, n1), 1)
    u, ref = s.solve(f), o.solve(f[3])
    _same_bits(s.solve, f, u)
    assert rel_err(u[3], ref) < 1e-9
    s.set_tensor(*o.tensor_setup())  # entries of the other class: no parity classes
    u = s.solve(f)
    _same_bits(s.solve, f, u)
    assert rel_err(u[3], ref) < 1e-12


def test_adi_solve(oracle):
    from rustpde_amd import Solver
    n0, n1, batch = 254, 252, 104
    print("case large batch adi", n0, n1, batch, flush=True)
    assert _large([(126, 127, 2, n1, batch)]) and _large([(125, 126, 2, n0 - 2, batch)])
    s = Solver(0, (DIRICHLET, n0), (NEUMANN, n1), (0.01, 0.02))
    f = _rand((batch, n0, n1), 2)
    u = s.solve(f)
    _same_bits(s.solve, f, u)
    assert rel_err(u[3], oracle.Solver("hholtz_adi", DIRICHLET, n0, NEUMANN, n1, [0.01, 0.02]).solve(f[3])) < 1e-12


# both products transposed (no fast transform along y), or one product beside the fast transform
@pytest.mark.parametrize("n1", [252, 257])
def test_space_operations(oracle, n1):
    from rustpde_amd import Space2
    n0, batch = 254, 104
    print("case large batch space", n0, n1, batch, flush=True)
    assert _large([(126, 127, 2, n1 - 2, batch)]) and _large([(127, 126, 2, n1 - 2, batch)])
    sp = Space2((DIRICHLET, n0), (NEUMANN, n1))
    for op, shape, deriv in (("forward", sp.shape_physical, None), ("backward", sp.shape_spectral, None),
                             ("to_ortho", sp.shape_spectral, None), ("from_ortho", sp.shape_ortho, None),
                             ("gradient", sp.shape_spectral, (1, 0)), ("gradient", sp.shape_spectral, (2, 0))):
        a = _rand((batch,) + tuple(shape), 3)
        call = (lambda v: sp.gradient(v, deriv, (1.0, 1.0))) if deriv else getattr(sp, op)
        got = call(a)
        _same_bits(call, a, got)
        kw = dict(deriv=deriv, scale=(1.0, 1.0)) if deriv else {}
        assert rel_err(got[3], oracle.space_apply(DIRICHLET, n0, NEUMANN, n1, op, a[3], **kw)) < 1e-12, (op, deriv)


def test_ensemble_step():
    """three products of a launch: the transforms of the fields' values and derivatives, d/dx of the pressure"""
    from rustpde_amd import Ensemble, Navier2D
    n, count = 254, 16
    print("case large batch ensemble", n, count, flush=True)
    assert _large([(127, 126, 2, n - 2, 3 * count), (127, 126, 2, n - 2, 3 * count), (127, 127, 2, n, count)])
    ra = [1e5 * (1 + i) for i in range(count)]
    e = Ensemble([(n, n, r, 1.0, 1e-3, 1.0, True) for r in ra])
    for i in range(count):
        e[i].set_velocity(0.1 + 0.01 * i, 1.0, 1.0)
        e[i].set_temperature(0.2, 1.0, 1.0)
    e.update(3)
    for i in (0, 7, count - 1):
        g = Navier2D.new(n, n, ra[i], 1.0, 1e-3, 1.0, True)
        g.set_option(g.OPT_DCT, 0)  # the group's y transforms
        g.set_velocity(0.1 + 0.01 * i, 1.0, 1.0)
        g.set_temperature(0.2, 1.0, 1.0)
        g.update(3)
        for a, b in ((e[i].temp, g.temp), (e[i].ux, g.ux), (e[i].uy, g.uy)):
            assert rel_err(a.vhat, b.vhat) < 1e-12, i
        assert rel_err(e[i].pres[0].vhat, g.pres[0].vhat) < 1e-10, i
        g.close()
    e.close()


@pytest.mark.parametrize("case", [(40, 940, 110), (39, 700, 131)])
def test_rows_of_eight_entries(case):
    from rustpde_amd import Solver
    n0, n1, batch = case
    print("case large batch rows", case, flush=True)
    per = ((n1 - 1) // 2 + 63) // 64
    pad = lambda i: i + i // 16  # noqa: E731
    assert 4 < per <= 8 and 4 * 2 * (pad(n1 + 6) + 1) * 8 <= 65536 and (n0 - 1) // 2 * (batch // 4) >= 500
    s = Solver(1, (NEUMANN, n0), (NEUMANN, n1), (0.01, 0.02))
    f = _rand((batch, n0, n1), 5)
    u = s.solve(f)
    for b in (0, 1, batch // 2, batch - 2, batch - 1):
        assert np.array_equal(u[b], s.solve(f[b])), b
