"""An error that another HIP call of the thread left behind is not this library's: calls that only wait and
copy succeed."""
import ctypes as C

import numpy as np
import pytest

from cleo_amd import abi
from cleo_amd import populations as P
from tests.helpers import SEED, make_domain

pytestmark = pytest.mark.gpu


def test_calls_after_a_foreign_error(gpu):
    print("case: waits and copies after a refused hipSetDevice", flush=True)
    g = make_domain(gpu, P.coal_breakup(SEED, ndims=(2, 2, 2), mean=20))
    L = gpu.lib
    nd, err, stats = C.c_uint64(), abi.Error(), abi.Stats()
    refs = np.zeros(9, dtype=np.uint32)
    calls = {
        "synchronize": lambda: L.cleo_synchronize(g.h),
        "ndomain": lambda: L.cleo_ndomain(g.h, C.byref(nd)),
        "get_error": lambda: L.cleo_get_error(g.h, C.byref(err)),
        "get_stats": lambda: L.cleo_get_stats(g.h, C.byref(stats)),
        "download_refs": lambda: L.cleo_download_refs(g.h, refs.ctypes.data_as(C.POINTER(C.c_uint32))),
        "set_rng_counter": lambda: L.cleo_set_rng_counter(g.h, C.c_uint64(1), C.c_uint64(0)),
    }
    for name, call in calls.items():
        assert L.hipSetDevice(1 << 20) != 0
        assert call() == 0, name
        L.hipGetLastError()
    assert nd.value == refs[8] > 0
