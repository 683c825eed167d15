"""GPU: runs of no steps."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _engines():
    from jaxabm_amd.programs.schelling import SchellingEngine
    from jaxabm_amd.programs.sir import SIRNetworkEngine
    from jaxabm_amd.programs.wealth import WealthEngine

    return {
        "wealth": lambda: WealthEngine(50, seed=3),
        "wealth_grid": lambda: WealthEngine(50_000, seed=3),
        "sir": lambda: SIRNetworkEngine(500, m=2, beta=0.2, n_seed_infected=10, seed=3),
        "schelling": lambda: SchellingEngine(20, 30, seed=3),
        "schelling_two_launches": lambda: SchellingEngine(200, 170, seed=3),
    }


@pytest.mark.parametrize("kind", ["wealth", "wealth_grid", "sir", "schelling",
                                  "schelling_two_launches"])
def test_run_of_no_steps(kind):
    """Empty records of the usual types, and the run that follows is that of an
    engine without it."""
    make = _engines()[kind]
    a, b = make(), make()
    none, want = a.run(0), b.run(6)
    got = a.run(6)
    if kind == "sir":
        none, want, got = (none,), (want,), (got,)
        np.testing.assert_array_equal(a.state_host(), b.state_host())
    for z, w, g in zip(none, want, got):
        assert z.shape == (0, *w.shape[1:]) and z.dtype == w.dtype
        np.testing.assert_array_equal(g, w)
    np.testing.assert_array_equal(a.rng, b.rng)
