"""Condensation over the whole range of radii: the ventilation factor's powers at both ends of a
binade, around its cap and where it is 1, against the oracle."""
import numpy as np
import pytest

from cleo_amd import populations as P
from tests.helpers import SEED, assert_supers_match, cond_params, make_domain

pytestmark = pytest.mark.gpu

RADII = {  # dimensionless, in micrometres
    "aerosol": (0.6, 2.0),
    "cloud": (2.0, 30.0),
    "rain": (30.0, 3000.0),
    "capped": (3000.0, 1e5),
}


@pytest.mark.parametrize("radii", list(RADII))
def test_condensation_radii(gpu, oracle, radii):
    print(f"case: condensation of radii {RADII[radii]}", flush=True)
    pop = P.condensation(SEED, ndims=(2, 2, 2), mean=200)
    lo, hi = RADII[radii]
    n = pop.n
    r = np.exp(np.random.default_rng(SEED).uniform(np.log(lo), np.log(hi), n))
    binade = np.exp2(np.floor(np.log2(r)))  # around powers of two of the radius in metres as well
    r[::5] = np.maximum(lo, binade[::5])
    r[1::5] = np.nextafter(np.maximum(lo, binade[1::5]), 0.0)
    r[2::5] = np.sqrt(2.0) * binade[2::5]
    pop.supers["radius"] = r
    pop.supers["msol"] = 0.1 * r ** 3  # a trace of solute in every drop
    g, o = make_domain(gpu, pop), make_domain(oracle, pop)
    for d in (g, o):
        assert d.condensation(cond_params(interval=100)) == 0, d.error()
    assert_supers_match(g.download(), o.download())
