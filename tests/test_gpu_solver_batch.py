"""The largest batch of a confined solve, 65535 right-hand sides, and one more, which is refused."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", [0, 1, 2])  # HholtzAdi, Hholtz, Poisson
def test_largest_batch(kind):
    from rustpde_amd import RbcError, Solver
    print("case largest batch", kind, flush=True)
    s = Solver(kind, (2, 8), (2, 9), (0.01, 0.02) if kind < 2 else (1.0, 1.0))
    f = np.random.default_rng(kind).standard_normal((65536,) + s.shape_in)
    with pytest.raises(RbcError, match="batch"):
        s.solve(f)
    u = s.solve(f[:65535])
    for b in (0, 1, 32767, 65534):
        assert np.array_equal(u[b], s.solve(f[b])), b
