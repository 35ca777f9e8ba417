"""Gridboxes whose pairs are shared out over several workgroups, and the end of a microphysics pass
(re-sort of the nulls, event count) by the last event's own kernel, one workgroup or two launches,
against the oracle (xi, order and refs bit-exact)."""
import numpy as np
import pytest

from cleo_amd import abi
from cleo_amd import populations as P
from tests.helpers import SEED, assert_supers_match, coll_params, make_domain

pytestmark = pytest.mark.gpu

SIZES = {
    "empty": [0, 3],
    "alone_3": [3],
    "alone_97": [97],
    "alone_513": [513],
    "alone_2049": [2049],
    "shares_8": [8191],
    "lds_full": [19200],
    "hbm": [19201],
    "shares_of_three": [6000, 2, 9001],
    "one_above_lds": [19500] + [300] * 30,
    "one_launch": [10] * 1000,
    "two_launches": [300] * 60,
}


@pytest.mark.parametrize("graph", [False, True])
@pytest.mark.parametrize("sizes", list(SIZES))
def test_collision_shares(gpu, oracle, sizes, graph):
    print(f"case: collisions of gridboxes {sizes}, graph {graph}", flush=True)
    counts = SIZES[sizes]
    pop = P.coal_breakup(SEED, ndims=(len(counts), 1, 1), mean=1.1 * sum(counts) / len(counts) + 20)
    pop.supers = {k: v[:sum(counts)].copy() for k, v in pop.supers.items()}
    pop.supers["sdgbxindex"] = np.repeat(np.arange(len(counts), dtype=np.uint32), counts)
    pop.supers["xi"][::3] = 1  # twins of multiplicity 1 become nulls
    first = coll_params(prob=abi.PROB_CONST, param=2e4 / max(counts), enact=abi.ENACT_COAL, interval=50)
    second = coll_params(prob=abi.PROB_LONG, enact=abi.ENACT_COAL, interval=100)
    g, o = make_domain(gpu, pop), make_domain(oracle, pop)
    for d in (g, o):
        d.rng_counter(SEED, 0)
        assert d.set_sdm_chain([abi.coll_process(first), abi.coll_process(second)]) == 0
    # a pass: both events, the first one again, the re-sort
    if graph:
        assert gpu.lib.cleo_run_steps_graph(g.h, 0, 100, 4) == 0, g.error()
    for t in range(0, 400, 100):
        if not graph:
            assert g.run_step(t, t + 100) == 0, g.error()
        assert o.run_step(t, t + 100) == 0, o.error()
    assert_supers_match(g.download(), o.download())
    assert np.array_equal(g.refs(), o.refs())
    for f in ("coll_pairs", "coll_events", "nulls"):
        assert g.stats()[f] == o.stats()[f], f
