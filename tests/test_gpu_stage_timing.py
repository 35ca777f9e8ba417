"""Stage timing of the fused motion, sort and condensation on a full store whose last gridboxes gain drops:
nothing outside the store is read, and drops, refs and State stay as they are."""
import ctypes as C

import numpy as np
import pytest

from cleo_amd import abi
from cleo_amd import populations as P
from tests.helpers import SEED, assert_state_match, assert_supers_match, cond_params, make_domain, motion_params, sdm_params

pytestmark = pytest.mark.gpu


def _windy(ndims, mean):
    """Drops in store order, as many as the context holds; the wind blows them to the last gridboxes."""
    pop = P.coupled(SEED, ndims=ndims, mean=mean)
    for f in ("vvel_lo", "vvel_hi"):
        pop.state[f] += 6.0
    last = pop.state["vvel_hi"].reshape(ndims[2], -1)
    last[-1] = 0.0  # and not out of them
    pop.periodic = (False, False, False)
    return pop


@pytest.mark.parametrize("tiles", [(1, 1, 1, 1, 1, 0, 0, 0, 0, 8), (1, 1, 1, 1, 3, 0, 0, 0, 0, 8)])
@pytest.mark.parametrize("ndims,mean", [((5, 4, 3), 20), ((16, 16, 16), 140)])
def test_fused_stage_leaves_the_store(gpu, oracle, ndims, mean, tiles):
    print(f"case: fused stage timed on {ndims} gridboxes of {mean}, tiles {tiles}", flush=True)
    pop = _windy(ndims, mean)
    g, o = make_domain(gpu, pop), make_domain(oracle, pop)
    assert gpu.lib.cleo_set_tiles(g.h, abi.ctypes_byref(abi.Tiles(*tiles))) == 0
    for d in (g, o):
        d.set_sdm(sdm_params(cond=cond_params(), motion=motion_params()))
    ms = C.c_float()
    assert gpu.lib.cleo_time_kernel(g.h, 3, 2, C.byref(ms)) == 0 and ms.value > 0
    assert_supers_match(g.download(), o.download(), exact_fp=True)
    assert_state_match(g.state(), o.state(), rtol=0.0)
    before = o.refs()
    assert np.array_equal(g.refs(), before)
    for d in (g, o):
        assert d.run_step(0, 100) == 0 and d.error()[0] == 0
    assert_supers_match(g.download(), o.download())
    assert_state_match(g.state(), o.state())
    after = o.refs()
    assert np.array_equal(g.refs(), after)
    assert (before[:-1] + np.diff(after)).max() > pop.n  # the old refs with the new counts lead out of the store
