"""The confined FP64 step's fused launches at their edges: grids around multiples of 16 points and of
16 coefficients of one parity, an axis pair of very different lengths, the y transforms as products and
(from 201 points) as fast transforms, ensembles large enough for the blocks of three fields, and the
divergence norm's row kernels.

Oracle tolerances 1e-12 as the other confined steps of these lengths; an ensemble and the step field by
field run the same sums as one instance of three fields, so they agree to 1e-14 and to the last bit."""
import numpy as np
import pytest

from helpers import compare, init_pair, rel_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(8, 8), (9, 17), (17, 10), (33, 34), (34, 66), (66, 35), (24, 201), (131, 20)])
def test_confined_sizes(oracle, shape):
    from rustpde_amd import Navier2D
    nx, ny = shape
    print("case confined %dx%d, 5 steps" % shape, flush=True)
    g = Navier2D.new(nx, ny, 1e4, 1.0, 5e-3, 1.0, True)
    o = oracle.Navier2D.new(nx, ny, 1e4, 1.0, 5e-3, 1.0, True)
    init_pair(g, o, nx, ny, False, 1e-2, 3, "uniform", velocity=(0.1, 1.0, 1.0))
    g.update(5)
    o.update(5)
    e = compare(g, o)
    for k in ("temp", "ux", "uy", "pres"):
        assert e[k] < 1e-12, (k, e)
    # the norm is that of a nearly divergence-free field: against the size of its terms
    assert abs(g.div_norm() - o.div_norm()) < 1e-12 * max(1.0, o.div_norm())
    assert not g.exit()
    g.temp.vhat, g.ux.vhat = g.temp.vhat, np.full_like(g.ux.vhat, np.nan)
    assert np.isnan(g.div_norm()) and g.exit()
    g.close()


@pytest.mark.parametrize("n,count", [(40, 24), (97, 13), (130, 2)])
def test_three_fields_in_a_block(n, count):
    from rustpde_amd import Ensemble, Navier2D, seeded
    print("case ensemble of %d at %d" % (count, n), flush=True)
    d = [(n, n, 1e4 * 1.2 ** i, 1.0, 0.2 / n, 1.0, True) for i in range(count)]
    seed = lambda nav, i: (nav.set_velocity(0.1, 1.0, 1.0), setattr(nav.temp, "v", seeded.interior_perturbation(
        n, n, 1e-2, 5 + i, kind="uniform", periodic=False)), nav.temp.forward())
    ens = Ensemble(d)
    for i in range(count):
        seed(ens[i], i)
    ens.update(4)
    for i in {0, count // 2, count - 1}:
        out = []
        for batch in (1, 0):
            s = Navier2D.new(*d[i])
            s.set_option(s.OPT_BATCH, batch)
            seed(s, i)
            s.update(4)
            out.append([f.vhat for f in (s.temp, s.ux, s.uy, s.pres[0])] + [s.div_norm()])
            s.close()
        assert all(np.array_equal(a, b) for a, b in zip(*out))
        mine = [f.vhat for f in (ens[i].temp, ens[i].ux, ens[i].uy, ens[i].pres[0])]
        for a, b in zip(mine, out[0]):
            assert rel_err(a, b) < 1e-14
        assert abs(ens[i].div_norm() - out[0][4]) < 1e-12 * max(1.0, out[0][4])
    ens.close()
