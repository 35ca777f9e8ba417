"""The re-sort of nulls at the end of a microphysics pass where a condensation follows the last collision
event and has applied its order to the store, against the oracle (xi, sdid, order and refs bit-exact)."""
import numpy as np
import pytest

from cleo_amd import abi
from cleo_amd import populations as P
from tests.helpers import (SEED, assert_state_match, assert_supers_match, coll_params, cond_params, make_domain,
                           motion_params)

pytestmark = pytest.mark.gpu

# one gridbox, the re-sort by one workgroup, and by two launches; 8192 of them have several gridboxes a workgroup
DOMAINS = {"alone": ((1, 1, 1), 300), "one_launch": ((4, 4, 3), 60), "two_launches": ((8, 8, 8), 40),
           "shared_out": ((32, 16, 16), 6)}


def _population(ndims, mean):
    pop = P.coupled(SEED, ndims=ndims, mean=mean)
    pop.supers["xi"][:] = 1 + np.arange(pop.n) % 3  # twins of multiplicity 1 become nulls
    return pop


@pytest.mark.parametrize("graph", [False, True])
@pytest.mark.parametrize("motion", [0, 100, 200])
@pytest.mark.parametrize("chain", ["colls_cond", "cond_twice"])
@pytest.mark.parametrize("domain", list(DOMAINS))
def test_condensation_after_the_last_event(gpu, oracle, domain, chain, motion, graph):
    print(f"case: nulls re-sorted after a condensation, {domain}, {chain}, motion {motion}, graph {graph}", flush=True)
    ndims, mean = DOMAINS[domain]
    pop = _population(ndims, mean)
    colls = coll_params(prob=abi.PROB_CONST, param=300.0, enact=abi.ENACT_COAL)  # most pairs are enacted
    procs = ([abi.coll_process(colls), abi.cond_process(cond_params())] if chain == "colls_cond" else
             [abi.cond_process(cond_params(interval=50)), abi.coll_process(colls)])
    span = motion if motion == 200 else 100
    g, o = make_domain(gpu, pop), make_domain(oracle, pop)
    for d in (g, o):
        d.rng_counter(SEED, 0)
        assert d.set_sdm_chain(procs, motion_params(interval=motion) if motion else None) == 0
    if graph:
        assert gpu.lib.cleo_run_steps_graph(g.h, 0, span, 3) == 0, g.error()
    for t in range(0, 3 * span, span):
        if not graph:
            assert g.run_step(t, t + span) == 0, g.error()
        assert o.run_step(t, t + span) == 0, o.error()
    assert g.error()[0] == 0 and o.error()[0] == 0
    assert o.stats()["nulls"] > 0
    # rounding may decide the convergence test of a drop at equilibrium, and one Newton iteration more or
    # less there moves its radius by the test's tolerance, 1e-8
    assert_supers_match(g.download(), o.download(), rtol=1e-7, what=chain)
    assert_state_match(g.state(), o.state(), rtol=1e-7, what=chain)
    assert np.array_equal(g.refs(), o.refs())
    for f in ("coll_events", "nulls", "sorts"):
        assert g.stats()[f] == o.stats()[f], f
