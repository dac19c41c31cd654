"""Batched confined solves whose row systems share a wavefront between four right-hand sides: batches of no
multiple of four, odd set counts, rows of two, four and eight entries a lane, and the same solves one at a
time.

Each right-hand side's row is solved by the same operations in both forms; the products before and after
them differ in their tile only, whose sums agree to the last bit, so the solutions do too."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("case", [(1, 1, 64, 30, 70), (1, 2, 65, 257, 67), (2, 2, 34, 130, 131), (1, 1, 130, 600, 33),
                                  (1, 2, 40, 1000, 110)])
def test_batch_of_rows(oracle, case):
    from rustpde_amd import Solver
    solver, kind, n0, n1, batch = case
    print("case batched rows", case, flush=True)
    c = (0.01, 0.02) if solver == 1 else (1.0, 1.0)
    s = Solver(solver, (kind, n0), (kind, n1), c)
    rng = np.random.default_rng(5)
    k = np.arange(n0)[:, None] + np.arange(n1)[None, :]
    f = rng.standard_normal((batch, n0, n1)) / (1.0 + k) ** 2
    u = s.solve(f)
    for b in (0, 1, batch // 2, batch - 2, batch - 1):
        assert np.array_equal(u[b], s.solve(f[b])), b
    o = oracle.Solver("hholtz" if solver == 1 else "poisson", kind, n0, kind, n1, list(c))
    if n0 * n1 < 20000:
        s.set_tensor(*o.tensor_setup())
        u, ref = s.solve(f), o.solve(f[batch - 1])
        assert np.abs(u[batch - 1] - ref).max() < 1e-12 * np.abs(ref).max()
