"""The parallel shuffle of the collisions at its edges: gridboxes around the team sizes, the LDS
capacity and the HBM path, against the oracle's serial Fisher-Yates (xi, order and refs bit-exact)."""
import ctypes as C

import numpy as np
import pytest

from cleo_amd import abi
from cleo_amd import populations as P
from tests.helpers import SEED, assert_supers_match, coll_params, injected_stream, make_domain

pytestmark = pytest.mark.gpu

SIZES = {
    "edges": [0, 1, 2, 3, 4, 5, 6, 0, 63, 64, 65, 127, 128, 129, 255, 256, 257, 1, 511, 512, 513, 635, 636, 637, 640],
    "one_of_2": [2],
    "one_of_1": [1],
    "team_256": [601, 2047, 1030],
    "team_1024": [2049],
    "team_1024_full": [7680, 7681],
    "hbm": [15361],
    "few_large": [5000] + [9] * 70 + [300, 0, 70, 1200],
}


def _population(counts, enact):
    pop = P.coal_breakup(SEED, ndims=(len(counts), 1, 1), mean=1.1 * sum(counts) / len(counts) + 20)
    assert pop.n >= sum(counts)
    pop.supers = {k: v[:sum(counts)].copy() for k, v in pop.supers.items()}
    pop.supers["sdgbxindex"] = np.repeat(np.arange(len(counts), dtype=np.uint32), counts)
    if enact == abi.ENACT_COAL:  # twins of multiplicity 1 become nulls
        pop.supers["xi"][::3] = 1
    return pop


@pytest.mark.parametrize("enact", [abi.ENACT_COALBURE, abi.ENACT_COAL])
@pytest.mark.parametrize("tiled", [0, 1])
@pytest.mark.parametrize("sizes", list(SIZES))
def test_team_shuffle(gpu, oracle, sizes, tiled, enact):
    print(f"case: shuffle of gridboxes {sizes}, tiled {tiled}, enactment {enact}", flush=True)
    pop = _population(SIZES[sizes], enact)
    g, o = make_domain(gpu, pop), make_domain(oracle, pop)
    assert gpu.lib.cleo_set_tiles(g.h, C.byref(abi.Tiles(1, 1, 1, 0, 0, 0, 0, 0, tiled))) == 0
    if enact == abi.ENACT_COAL:
        p = coll_params(prob=abi.PROB_CONST, param=1e-3, enact=enact)  # most pairs are enacted
    else:
        p = coll_params(prob=abi.PROB_LONG, enact=enact)
    js, phis = injected_stream(o.refs(), np.random.default_rng(3))
    for d in (g, o):
        d.rng_injected(js, phis)
        assert d.collisions(p) == 0
        d.rng_counter(SEED, 5)
    assert_supers_match(g.download(), o.download(), what="injected")
    for _ in range(3):  # the orders of the later events compose
        assert g.collisions(p) == 0
        assert o.collisions(p) == 0
    assert_supers_match(g.download(), o.download(), what="counter")
    assert np.array_equal(g.refs(), o.refs())
    for f in ("coll_pairs", "coll_events", "nulls"):
        assert g.stats()[f] == o.stats()[f], f


def test_tiles_with_large_gridboxes(gpu, oracle):
    print("case: tiles of a large domain, gridboxes above 255 drops and above the tile's LDS", flush=True)
    counts = np.full(75000, 3)
    counts[64:128] = 150  # a tile whose permutations overflow
    counts[[300, 301, 400, 512, 700, 74999]] = [256, 636, 637, 700, 255, 2]
    pop = _population(counts.tolist(), abi.ENACT_COAL)
    g, o = make_domain(gpu, pop), make_domain(oracle, pop)
    assert gpu.lib.cleo_set_tiles(g.h, C.byref(abi.Tiles(1, 1, 1, 0, 0, 0, 0, 0, 1))) == 0
    p = coll_params(prob=abi.PROB_CONST, param=1e-3, enact=abi.ENACT_COAL)
    for d in (g, o):
        d.rng_counter(SEED, 0)
        assert d.collisions(p) == 0 and d.collisions(p) == 0
    assert_supers_match(g.download(), o.download(), what="tiles")
    assert g.stats()["coll_events"] == o.stats()["coll_events"] and g.stats()["nulls"] == o.stats()["nulls"]
