"""A download that fails half way: the fields copied before the failure are whole when the call returns, and
nothing is written afterwards."""
import ctypes as C

import numpy as np
import pytest
import torch

from cleo_amd import abi

pytestmark = pytest.mark.gpu


def test_download_without_the_last_field(gpu):
    n = 1 << 24
    print(f"case: download of {n} drops without sdid", flush=True)
    g = abi.Domain(gpu, n, (1, 1, 1), [0.0, 1.0], [0.0, 1.0], [0.0, 1.0])
    dtypes = {f: (torch.int32 if f == "sdgbxindex" else torch.int64 if f in ("xi", "sdid") else torch.float64)
              for f, _ in abi.SupersSoA._fields_}
    src = {f: torch.arange(1, n + 1, device="cuda").to(t) if f != "sdgbxindex" else
           torch.zeros(n, device="cuda", dtype=t) for f, t in dtypes.items()}
    out = {f: torch.full((n,), -1, dtype=t).pin_memory() for f, t in dtypes.items()}

    def soa(tensors):
        s = abi.SupersSoA()
        for name, ctype in abi.SupersSoA._fields_:
            setattr(s, name, C.cast(C.c_void_p(tensors[name].data_ptr()), ctype))
        return s

    torch.cuda.synchronize()
    assert gpu.lib.cleo_upload_supers_device(g.h, C.byref(soa(src)), n) == 0
    s = soa(out)
    setattr(s, "sdid", None)
    rc = gpu.lib.cleo_download_supers(g.h, C.byref(s), None, None)
    last = [int(out[f][-1]) for f in ("radius", "msol")]  # read at once, before anything else waits
    assert rc == abi.CLEO_E_HIP and last == [n, n]
    gpu.lib.hipGetLastError()
    for f in ("coord3", "xi", "msol"):
        assert torch.equal(out[f], torch.arange(1, n + 1).to(dtypes[f])), f
    assert np.all(out["sdid"].numpy() == -1)
