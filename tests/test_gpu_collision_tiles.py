"""Collisions by tiles of 64 gridboxes (domains of 75000 gridboxes and more): every kernel, enactment and flag
with kinetic energies and without, injected and counter streams, nulls, against the oracle (xi, order and
refs bit-exact).  Among the small gridboxes are ones of 255 to 700 drops, which the whole wave shuffles."""
import numpy as np
import pytest

from cleo_amd import abi
from cleo_amd import populations as P
from tests.helpers import SEED, assert_supers_match, coll_params, injected_stream, make_domain

pytestmark = pytest.mark.gpu

GK, SIMMEL, YAU = abi.TV_ROGERS_GK, abi.TV_SIMMEL, abi.TV_ROGERS_YAU
CASES = {
    "golovin": dict(prob=abi.PROB_GOLOVIN, param=0.0, enact=abi.ENACT_COAL),
    "long_breakup": dict(prob=abi.PROB_LONG, enact=abi.ENACT_BREAKUP),
    "long_coalbure": dict(prob=abi.PROB_LONG, enact=abi.ENACT_COALBURE),
    "lowlist_coal": dict(prob=abi.PROB_LOWLIST_COAL, prob_tv=SIMMEL, enact=abi.ENACT_COAL),
    "lowlist_bu_cke": dict(prob=abi.PROB_LOWLIST_BU, prob_tv=SIMMEL, enact=abi.ENACT_BREAKUP,
                           nfrags_kind=abi.NFRAGS_CKE, nfrags_tv=SIMMEL),
    "su_cke": dict(prob=abi.PROB_LONG, enact=abi.ENACT_COALBURE, nfrags_kind=abi.NFRAGS_CKE, nfrags_tv=YAU,
                   flag_kind=abi.FLAG_SU, flag_tv=SIMMEL),
    "ts": dict(prob=abi.PROB_LONG, enact=abi.ENACT_COALBURE, flag_kind=abi.FLAG_TS, flag_tv=GK),
    "straub": dict(prob=abi.PROB_LONG, enact=abi.ENACT_COALBURE, flag_kind=abi.FLAG_STRAUB, flag_tv=SIMMEL),
}


def _population(nulls):
    counts = np.arange(75003) % 6
    counts[64:128] = 150  # a tile whose permutations overflow
    counts[[300, 301, 400, 512, 700, 75002]] = [255, 256, 637, 700, 129, 2]
    n = int(counts.sum())
    pop = P.coal_breakup(SEED, ndims=(len(counts), 1, 1), mean=4)
    rng = np.random.default_rng(SEED + 1)
    assert pop.n >= n
    pop.supers = {k: v[:n].copy() for k, v in pop.supers.items()}
    pop.supers["sdgbxindex"] = np.repeat(np.arange(len(counts), dtype=np.uint32), counts)
    wet = np.exp(rng.uniform(np.log(20.0), np.log(2500.0), n))  # both sides of every flag's boundaries
    pop.supers["radius"] = np.maximum(wet, pop.supers["radius"])
    pop.state["volume"] *= 0.1  # a sixth to a third of the pairs are enacted
    if nulls:
        pop.supers["xi"][:] = 1 + np.arange(n) % 3
        pop.state["volume"] *= 1e-9
    return pop


@pytest.mark.parametrize("stream", ["injected", "counter"])
@pytest.mark.parametrize("case", list(CASES) + ["lowlist_coal_nulls"])
def test_tiles(gpu, oracle, case, stream):
    print(f"case: collisions by tiles, {case}, {stream}", flush=True)
    pop = _population(case.endswith("nulls"))
    p = coll_params(**CASES[case.replace("_nulls", "")])
    g, o = make_domain(gpu, pop), make_domain(oracle, pop)
    rng = np.random.default_rng(7)
    for d in (g, o):
        d.rng_counter(SEED, 3)
    for step in range(2):  # (the second event's order composes with the first's)
        if stream == "injected":
            js, phis = injected_stream(o.refs(), rng)
            for d in (g, o):
                d.rng_injected(js, phis)
        for d in (g, o):
            assert d.collisions(p) == 0
    assert g.error()[0] == 0 and o.error()[0] == 0
    assert o.stats()["coll_events"] > 1000 and (o.stats()["nulls"] > 0 or not case.endswith("nulls"))
    assert_supers_match(g.download(), o.download(), what=case)
    assert np.array_equal(g.refs(), o.refs())
    for f in ("coll_pairs", "coll_events", "nulls"):
        assert g.stats()[f] == o.stats()[f], f
