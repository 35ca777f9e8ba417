"""The generic sort at the edges of its tiles and digits, with and without a context, against a stable
sort of the keys: every field bit for bit, and the refs."""
import ctypes as C

import numpy as np
import pytest
import torch

from cleo_amd import abi

pytestmark = pytest.mark.gpu


def _drops(n, ngbx, sorted_keys, rng):
    key = rng.integers(0, ngbx, n).astype(np.uint32)
    key[rng.random(n) < 0.05] = abi.OOB
    key[rng.random(n) < 0.05] = ngbx
    if sorted_keys:
        key = np.sort(key)
    sup = {f: rng.random(n) for f in ("coord3", "coord1", "coord2", "radius", "msol")}
    sup.update(sdgbxindex=key, xi=rng.integers(1, 1 << 60, n).astype(np.uint64), sdid=np.arange(n, dtype=np.uint64))
    return sup


def _check(out, refs, sup, ngbx):
    key = np.minimum(sup["sdgbxindex"].astype(np.int64), ngbx)
    at = np.argsort(key, kind="stable")
    for f in sup:
        assert np.array_equal(out[f], sup[f][at]), f
    assert np.array_equal(refs, np.searchsorted(key[at], np.arange(ngbx + 1)))


@pytest.mark.parametrize("sorted_keys", [False, True])
@pytest.mark.parametrize("n", [1, 63, 64, 65, 2047, 2048, 2049, 8192 + 7, 300001])
@pytest.mark.parametrize("ngbx", [1, 2, 255, 256, 511, 65535, 65536, 1 << 20])
def test_radix_edges(gpu, n, ngbx, sorted_keys):
    print(f"case: radix sort of {n} drops over {ngbx} gridboxes, sorted {sorted_keys}", flush=True)
    sup = _drops(n, ngbx, sorted_keys, np.random.default_rng(n + ngbx))
    signed = {k: v.view({"uint32": np.int32, "uint64": np.int64}.get(str(v.dtype), v.dtype)) for k, v in sup.items()}
    tin = {k: torch.from_numpy(v).cuda() for k, v in signed.items()}
    tout = {k: torch.empty_like(v) for k, v in tin.items()}
    refs = torch.empty(ngbx + 1, dtype=torch.int32, device="cuda")
    views = []
    for t in (tin, tout):
        s = abi.SupersSoA()
        for name, ctype in abi.SupersSoA._fields_:
            setattr(s, name, C.cast(C.c_void_p(t[name].data_ptr()), ctype))
        views.append(s)
    torch.cuda.synchronize()
    fn = gpu.lib.cleo_sort_supers_noalloc
    fn.argtypes = [C.c_void_p, C.c_void_p, C.c_void_p, C.c_uint64, C.c_uint32, C.c_void_p]
    assert fn(C.byref(views[0]), C.byref(views[1]), C.c_void_p(refs.data_ptr()), n, ngbx, None) == 0
    torch.cuda.synchronize()
    _check({k: v.cpu().numpy().view(sup[k].dtype) for k, v in tout.items()}, refs.cpu().numpy(), sup, ngbx)
    if ngbx <= 65536:
        d = abi.Domain(gpu, n, (ngbx, 1, 1), np.arange(ngbx + 1.0), [0.0, 1.0], [0.0, 1.0])
        d.upload(sup)
        _check(d.download(), d.refs(), sup, ngbx)
