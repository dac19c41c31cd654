"""An ensemble with an instance whose parameters mean nothing (Ra negative or NaN: a parameter sweep gone
too far) is made and advanced: that instance's fields are NaN and exit() says so, the others of its group are
those of a group without it, bit for bit, wherever it stands in the group."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _run(ra, n):
    from rustpde_amd import Ensemble
    e = Ensemble([(n, n, r, 1.0, 1e-2, 1.0, True) for r in ra])
    for i in range(len(ra)):
        e[i].set_velocity(0.1, 1.0, 1.0)
        e[i].set_temperature(0.1 * (1 + i), 1.0, 1.0)
    e.update(3)
    out = [([f.vhat for f in (e[i].temp, e[i].ux, e[i].uy, e[i].pres[0])], e[i].exit()) for i in range(len(ra))]
    e.close()
    return out


@pytest.mark.filterwarnings("ignore:invalid value:RuntimeWarning")
@pytest.mark.parametrize("n", [32, 33])
@pytest.mark.parametrize("bad", [-1.0, float("nan")])
@pytest.mark.parametrize("at", [0, 1, 2])
def test_instance_without_meaning(n, bad, at):
    print("case ensemble invalid", n, bad, at, flush=True)
    ra = [1e4, 2e4, 3e4]
    good = _run(ra, n)
    got = _run(ra[:at] + [bad] + ra[at + 1:], n)
    for i in range(3):
        if i == at:
            assert got[i][1] and not np.isfinite(got[i][0][1]).any()
            continue
        assert not got[i][1]
        for a, b in zip(got[i][0], good[i][0]):
            assert np.array_equal(a, b), i
