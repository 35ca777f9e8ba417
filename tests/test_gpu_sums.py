"""Per-gridbox sums at the edges of their tiles: from one gridbox per wave to 64, empty gridboxes and a
last tile that is not full, against the oracle (the mass moments bit-exact: same order, same roundings)."""
import numpy as np
import pytest

from cleo_amd import abi
from cleo_amd import populations as P
from tests.helpers import SEED, assert_state_match, assert_supers_match, cond_params, make_domain, motion_params, sdm_params

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("variant", [0, 1])
@pytest.mark.parametrize("ndims,mean", [((3, 3, 3), 700), ((2, 3, 3), 513), ((5, 4, 3), 130), ((9, 5, 3), 3), ((41, 20, 23), 9)])
def test_sums_over_tiles(gpu, oracle, ndims, mean, variant):
    print(f"case: sums of {ndims} gridboxes of {mean}, variant {variant}", flush=True)
    pop = P.coupled(SEED, ndims=ndims, mean=mean)
    keep = pop.supers["sdgbxindex"] != 1  # an empty gridbox
    pop.supers = {k: v[keep].copy() for k, v in pop.supers.items()}
    g, o = make_domain(gpu, pop), make_domain(oracle, pop)
    t = abi.Tiles(1, 1, 1, variant, variant, 0, 0, 0, 0, 8 * variant)
    assert gpu.lib.cleo_set_tiles(g.h, abi.ctypes_byref(t)) == 0
    for rain in (False, True):
        for a, b in zip(g.mass_moments(rain), o.mass_moments(rain)):
            assert np.array_equal(a, b)
    for d in (g, o):
        d.set_sdm(sdm_params(cond=cond_params(), motion=motion_params()))
        assert d.run_step(0, 100) == 0
    assert_supers_match(g.download(), o.download(), what="sums")
    assert_state_match(g.state(), o.state(), what="sums")
