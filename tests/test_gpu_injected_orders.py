"""Injected shuffle indices that put all swaps of a gridbox on one list, or all its places in one chain,
against the oracle's serial Fisher-Yates (xi, order and refs bit-exact)."""
import numpy as np
import pytest

from cleo_amd import abi
from cleo_amd import populations as P
from tests.helpers import SEED, assert_supers_match, coll_params, make_domain

pytestmark = pytest.mark.gpu

SIZES = {
    "wave": [90] * 20 + [0, 1, 2, 700],
    "large_for_a_wave": [40] * 900 + [3000],  # its lists in HBM
    "workgroup": [513],
    "one_each": [1500] * 600,
    "shares": [8192],
    "lds_full": [19200],
    "hbm": [19201],
    "far_above_lds": [150000],
}
# swap iter (from n-1 down to 1) with the element at:
INDEX = {
    "first": lambda it: 0 * it,
    "the_7th": lambda it: np.minimum(it, 6),
    "one_below": lambda it: it - 1,
    "itself": lambda it: it,
    "half": lambda it: it // 2,
    "two_places": lambda it: np.minimum(it, 1 + it % 2),
    "within_the_budget": lambda it: it // 300 * 300,
}


@pytest.mark.parametrize("index", list(INDEX))
@pytest.mark.parametrize("sizes", list(SIZES))
def test_injected_order(gpu, oracle, sizes, index):
    print(f"case: injected indices {index} in gridboxes {sizes}", flush=True)
    counts = SIZES[sizes]
    pop = P.coal_breakup(SEED, ndims=(len(counts), 1, 1), mean=1.1 * sum(counts) / len(counts) + 20)
    pop.supers = {k: v[:sum(counts)].copy() for k, v in pop.supers.items()}
    pop.supers["sdgbxindex"] = np.repeat(np.arange(len(counts), dtype=np.uint32), counts)
    js = np.concatenate([INDEX[index](np.arange(n - 1, 0, -1)) for n in counts if n >= 2] + [np.zeros(0, int)])
    phis = np.random.default_rng(3).random(sum(2 * (n // 2) for n in counts))
    p = coll_params(prob=abi.PROB_CONST, param=1e-3, enact=abi.ENACT_COAL)
    g, o = make_domain(gpu, pop), make_domain(oracle, pop)
    for d in (g, o):
        d.rng_injected(js.astype(np.uint32), phis)
        assert d.collisions(p) == 0
        d.rng_counter(SEED, 5)  # the next event's order composes with it
        assert d.collisions(p) == 0
    assert g.error()[0] == 0 and o.error()[0] == 0
    assert_supers_match(g.download(), o.download(), what=index)
    assert np.array_equal(g.refs(), o.refs())
    for f in ("coll_pairs", "coll_events", "nulls"):
        assert g.stats()[f] == o.stats()[f], f
