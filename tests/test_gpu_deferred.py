"""Deferred Newton solves: the drops set aside by their workgroup give what the undisturbed solves give,
whether the workgroup solves them at its end (small stores) or a second launch does (6M drops and more)."""
import ctypes as C

import pytest
import torch

from cleo_amd import abi
from cleo_amd import populations as P
from tests.helpers import SEED, assert_state_match, assert_supers_match, cond_params, motion_params, sdm_params

pytestmark = pytest.mark.gpu


def _step(gpu, ndims, mean, motion, tiles):
    sup, st, halves = P.coupled_device(torch, torch.device("cuda:0"), seed=SEED, ndims=ndims, spacing_m=25.0, mean=mean)
    torch.cuda.synchronize()
    n = sup["xi"].numel()
    d = abi.Domain(gpu, n, ndims, *halves)
    s = abi.SupersSoA()
    for name, ctype in abi.SupersSoA._fields_:
        setattr(s, name, C.cast(C.c_void_p(sup[name].data_ptr()), ctype))
    d.check(gpu.lib.cleo_upload_supers_device(d.h, C.byref(s), n), "upload")
    d.ntot = n
    d.set_state(st)
    d.set_solute(*P.solute_dimless(P.AMMONIUM_SULPHATE))
    assert gpu.lib.cleo_set_tiles(d.h, C.byref(abi.Tiles(*tiles))) == 0
    d.record_niters(True)
    d.set_sdm(sdm_params(cond=cond_params(), motion=motion_params() if motion else None))
    assert d.run_step(0, 100) == 0
    return d.download(), d.state(), d.niters(), d.stats()


@pytest.mark.parametrize("motion", [False, True])
@pytest.mark.parametrize("ndims,mean", [((3, 3, 2), 21), ((20, 16, 8), 64), ((50, 50, 40), 62)])
def test_deferred_equals_undeferred(gpu, ndims, mean, motion):
    print(f"case: deferred solves on {ndims} gridboxes of {mean}, motion {motion}", flush=True)
    base = _step(gpu, ndims, mean, motion, (1, 1, 1, 1, 1, 0, 0, 0, 0, 0))
    for defer, waves, variant in ((2, 0, 1), (6, 0, 3), (4, 4, 1)):
        if waves and ndims[0] == 50:
            waves = 4096
        out = _step(gpu, ndims, mean, motion, (1, 1, 1, 1, variant, waves, 0, 0, 0, defer))
        assert_supers_match(base[0], out[0], exact_fp=True, what=f"defer {defer}")
        assert_state_match(base[1], out[1], rtol=0.0, what=f"defer {defer}")
        assert (base[2] == out[2]).all()
        for f in ("cond_drops", "newton_iters", "substep_drops"):
            assert base[3][f] == out[3][f], f
