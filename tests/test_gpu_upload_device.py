"""cleo_upload_supers_device with arrays that the sort's kernels cannot read directly: a null field is an
error that leaves the context usable, pinned host arrays are copied."""
import ctypes as C

import numpy as np
import pytest
import torch

from cleo_amd import abi
from cleo_amd import populations as P
from tests.helpers import SEED, assert_supers_match, make_domain

pytestmark = pytest.mark.gpu

N = 5000
SIGNED = {"uint32": np.int32, "uint64": np.int64}


def _population():
    pop = P.coal_breakup(SEED, ndims=(4, 4, 4), mean=100)
    rng = np.random.default_rng(SEED)
    at = rng.permutation(pop.n)[:N]
    pop.supers = {k: np.ascontiguousarray(v[at]) for k, v in pop.supers.items()}
    return pop


def _soa(tensors):
    s = abi.SupersSoA()
    for name, ctype in abi.SupersSoA._fields_:
        setattr(s, name, C.cast(C.c_void_p(tensors[name].data_ptr()), ctype))
    return s


def _tensors(pop, pinned):
    t = {k: torch.from_numpy(v.view(SIGNED.get(str(v.dtype), v.dtype)).copy()) for k, v in pop.supers.items()}
    return {k: v.pin_memory() if pinned else v.cuda() for k, v in t.items()}


@pytest.mark.parametrize("field", [f for f, _ in abi.SupersSoA._fields_])
def test_null_field_is_an_error(gpu, oracle, field):
    print(f"case: upload from device arrays without {field}", flush=True)
    pop = _population()
    g, o = abi.Domain(gpu, N, pop.ndims, *pop.halves), make_domain(oracle, pop)
    t = _tensors(pop, False)
    torch.cuda.synchronize()
    s = _soa(t)
    setattr(s, field, None)
    assert gpu.lib.cleo_upload_supers_device(g.h, C.byref(s), N) == abi.CLEO_E_HIP
    assert gpu.lib.cleo_upload_supers_device(g.h, C.byref(s), 0) == 0  # no drops, nothing to read
    assert gpu.lib.cleo_upload_supers_device(g.h, C.byref(_soa(t)), N) == 0
    g.ntot = N
    assert_supers_match(g.download(), o.download(), exact_fp=True)
    assert np.array_equal(g.refs(), o.refs())


@pytest.mark.parametrize("pinned", [False, True])
def test_device_and_pinned_arrays(gpu, oracle, pinned):
    print(f"case: upload from device arrays, pinned {pinned}", flush=True)
    pop = _population()
    g, o = abi.Domain(gpu, N, pop.ndims, *pop.halves), make_domain(oracle, pop)
    t = _tensors(pop, pinned)
    torch.cuda.synchronize()
    assert gpu.lib.cleo_upload_supers_device(g.h, C.byref(_soa(t)), N) == 0
    g.ntot = N
    assert_supers_match(g.download(), o.download(), exact_fp=True)
    assert np.array_equal(g.refs(), o.refs())
