"""Motion and sort on periodic axes of one and two gridboxes, where steps in both directions lead to the
same neighbour: every motion variant against the oracle."""
import pytest

from cleo_amd import abi
from cleo_amd import populations as P
from tests.helpers import SEED, assert_state_match, assert_supers_match, cond_params, make_domain, motion_params, sdm_params

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("variant", [0, 1, 2, 3])
@pytest.mark.parametrize("ndims", [(5, 1, 1), (4, 2, 1), (4, 1, 2), (3, 2, 2), (1, 2, 3), (6, 3, 1)])
def test_narrow_periodic_axes(gpu, oracle, ndims, variant):
    print(f"case: motion on {ndims}, variant {variant}", flush=True)
    pop = P.coupled(SEED, ndims=ndims, mean=70, wmax_mps=6.0)
    pop.state["uvel_lo"] += 5.0  # every step some drops wrap around, in both directions
    pop.state["uvel_hi"] += 5.0
    pop.state["vvel_lo"] -= 4.0
    pop.state["vvel_hi"] -= 4.0
    g, o = make_domain(gpu, pop), make_domain(oracle, pop)
    assert gpu.lib.cleo_set_tiles(g.h, abi.ctypes_byref(abi.Tiles(1, 1, 1, 1, variant, 0, 0, 0, 0, 8))) == 0
    for cond in (None, cond_params()):
        for d in (g, o):
            d.set_sdm(sdm_params(cond=cond, motion=motion_params()))
        for step in range(4):
            assert g.run_step(100 * step, 100 * step + 100) == 0
            assert o.run_step(100 * step, 100 * step + 100) == 0
        assert g.error()[0] == 0 and o.error()[0] == 0
        assert_supers_match(g.download(), o.download(), what=f"narrow {cond is not None}")
    assert (g.refs() == o.refs()).all()
    assert_state_match(g.state(), o.state(), what="narrow")
