"""The dense x operators as parity classes (blocks, folds of mirrored points, no structure) at the
edges of their tiles and slabs: sizes around multiples of 32 and 64 rows and of 32 inputs per
class, one column and ragged column counts, batches that select the larger tile, and an operator
whose entries do not separate (a solver's eigenvectors set from outside).

Oracle tolerance 1e-12 of the largest value, as the other tests of these operations."""
import numpy as np
import pytest

from conftest import rel_err

pytestmark = pytest.mark.gpu

CASES = [  # (kind0, n0, n1, batch)
    (0, 6, 6, 1), (1, 7, 9, 2), (2, 33, 6, 1), (1, 34, 33, 3), (0, 63, 31, 2), (2, 64, 65, 1), (1, 65, 33, 2),
    (0, 66, 40, 1), (1, 127, 7, 2), (2, 130, 129, 1), (0, 131, 24, 1), (1, 258, 34, 1), (1, 130, 130, 40),
    (0, 97, 200, 64),
]


def _rand(shape, seed):
    rng = np.random.default_rng(seed)
    k = np.arange(shape[-2])[:, None] + np.arange(shape[-1])[None, :]
    return rng.standard_normal(shape) / (1.0 + k) ** 2


@pytest.mark.parametrize("case", CASES)
def test_x_operators(oracle, case):
    from rustpde_amd import Space2
    k0, n0, n1, batch = case
    print("case x operators", case, flush=True)
    sp = Space2((k0, n0), (1, n1))
    pick = sorted({0, batch // 2, batch - 1})
    for op, shp, kw in (("forward", sp.shape_physical, {}), ("backward", sp.shape_spectral, {}),
                        ("to_ortho", sp.shape_spectral, {}), ("from_ortho", sp.shape_ortho, {}),
                        ("gradient", sp.shape_spectral, {"deriv": (1, 0)}),
                        ("gradient", sp.shape_spectral, {"deriv": (2, 0)})):
        a = _rand((batch,) + shp, 7)
        got = sp.gradient(a, kw["deriv"], (1.0, 1.0)) if kw else getattr(sp, op)(a)
        for b in pick:
            ref = oracle.space_apply(k0, n0, 1, n1, op, a[b], **(dict(kw, scale=(1.0, 1.0)) if kw else {}))
            assert rel_err(got[b], ref) < 1e-12, (op, kw, b, rel_err(got[b], ref))


@pytest.mark.parametrize("case", [("hholtz", 1, 34, 20, 3), ("hholtz", 2, 67, 33, 2), ("poisson", 2, 66, 40, 1),
                                  ("hholtz_adi", 1, 65, 36, 3), ("hholtz", 1, 40, 30, 70)])
def test_solves_with_separating_and_mixed_eigenvectors(oracle, case):
    """The product's own eigenvectors separate by parity; the oracle's, set through the tensor's pub
    fields, hold rounding in the other class and take the undivided product."""
    from rustpde_amd import Solver
    kind, k0, n0, n1, batch = case
    print("case solve classes", case, flush=True)
    c = (0.01, 0.02) if kind != "poisson" else (1.0, 1.0)
    g = Solver({"hholtz_adi": 0, "hholtz": 1, "poisson": 2}[kind], (k0, n0), (1, n1), c)
    o = oracle.Solver(kind, k0, n0, 1, n1, list(c))
    f = _rand((batch,) + g.shape_in, 3)
    ref = np.stack([o.solve(f[b]) for b in range(batch)])
    own = g.solve(f)
    t = o.tensor_setup()
    if t is not None:
        lam, fwd, bwd = g.tensor_setup()
        if fwd is not None:  # exact zeros between the classes
            cls = np.abs(bwd[1::2]).max(axis=0) > 0
            assert not np.any(bwd[0::2][:, cls]) and not np.any(bwd[1::2][:, ~cls])
        # two eigen-decompositions: the eigenvalues agree to 1e-12 at these sizes, the solutions to 1e-9
        assert rel_err(own, ref) < 1e-9, rel_err(own, ref)
        g.set_tensor(*t)
        assert rel_err(g.solve(f), ref) < 1e-12, rel_err(g.solve(f), ref)
    else:
        assert rel_err(own, ref) < 1e-12, rel_err(own, ref)
