"""Per-gridbox sums by rows where the dispatch takes them, with one sum and two: empty and tiny gridboxes,
lengths around the rows' 31 values, a last tile that is not full, and gridboxes whose nulls, left by a
collision event before the condensation, are not summed."""
import numpy as np
import pytest

from cleo_amd import abi
from cleo_amd import populations as P
from tests.helpers import (SEED, assert_state_match, assert_supers_match, coll_params, cond_params, make_domain,
                           motion_params)

pytestmark = pytest.mark.gpu


def _population(ndims):
    pop = P.coupled(SEED, ndims=ndims, mean=165)
    g = pop.supers["sdgbxindex"].astype(np.int64)
    nth = np.arange(len(g)) - np.searchsorted(g, g)  # the drop's number in its gridbox
    most = np.full(int(np.prod(ndims)), 1 << 20)
    most[[0, 5, 17, 40, 41, 42, 43, 44, 45, 46]] = [0, 1, 0, 30, 31, 32, 61, 62, 63, 2]
    keep = nth < most[g]
    pop.supers = {k: v[keep].copy() for k, v in pop.supers.items()}
    return pop


@pytest.mark.parametrize("ndims,chain", [((32, 16, 17), "motion"), ((33, 31, 17), "alone"), ((33, 31, 17), "nulls")])
def test_sums_by_rows(gpu, oracle, ndims, chain):
    print(f"case: sums by rows of {ndims} gridboxes, {chain}", flush=True)
    pop = _population(ndims)
    procs = [abi.cond_process(cond_params())]
    if chain == "nulls":
        pop.supers["xi"][:] = 1 + np.arange(pop.n) % 3
        procs.insert(0, abi.coll_process(coll_params(prob=abi.PROB_CONST, param=300.0, enact=abi.ENACT_COAL)))
    g, o = make_domain(gpu, pop), make_domain(oracle, pop)
    for d in (g, o):
        d.rng_counter(SEED, 0)
        assert d.set_sdm_chain(procs, motion_params() if chain == "motion" else None) == 0
        assert d.run_step(0, 100) == 0 and d.error()[0] == 0
    assert (o.stats()["nulls"] > 0) == (chain == "nulls")
    assert_supers_match(g.download(), o.download(), what=chain)
    assert_state_match(g.state(), o.state(), what=chain)
