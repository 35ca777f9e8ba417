"""The sample order of a training whose seed makes the xorshift64 state 0: every index drawn is 0, and all
swaps are with the first sample."""
import ctypes as C

import numpy as np
import pytest
import torch

from cleo_amd import abi

pytestmark = pytest.mark.gpu

ZERO_STATE_SEED = 0xD1B54A32D192ED03


@pytest.mark.parametrize("n", [64, 257, 1000, 100003])
def test_order_of_the_zero_state(gpu, n):
    """With a learning rate of 0 the reported loss is that of the last batch under the initial weights: it
    must be the loss of the samples the serial shuffle puts there."""
    print(f"case: sample order of {n} samples from the zero state", flush=True)
    batch = max(1, n // 7)
    perm = list(range(n))
    for i in range(n - 1, 0, -1):
        perm[i], perm[0] = perm[0], perm[i]
    order = list(range(max(1, n // batch)))
    for b in range(len(order) - 1, 0, -1):
        order[b], order[0] = order[0], order[b]
    last = torch.tensor(perm[order[-1] * batch:order[-1] * batch + batch], device="cuda")
    rng = np.random.default_rng(n)
    x = torch.zeros((n, 8), device="cuda", dtype=torch.float32)
    x[:, :6] = torch.from_numpy(rng.normal(size=(n, 6)).astype(np.float32)).cuda()
    y = torch.from_numpy(rng.normal(size=n).astype(np.float32) * 3).cuda()
    xb, yb = x[last].contiguous(), y[last].contiguous()
    torch.cuda.synchronize()
    d = abi.Domain(gpu, 64, (1, 1, 1), [0.0, 1.0], [0.0, 1.0], [0.0, 1.0])
    got, want = C.c_float(), C.c_float()
    grad = np.zeros(abi.MLP_NPARAMS, dtype=np.float32)
    tp = abi.MLPTrainParams(1, batch, 0.0, 0.9, 0.999, 1e-8, ZERO_STATE_SEED)
    d.check(gpu.lib.cleo_mlp_train(d.h, x.data_ptr(), y.data_ptr(), n, C.byref(tp), C.byref(got)), "train")
    d.check(gpu.lib.cleo_mlp_loss_grad(d.h, xb.data_ptr(), yb.data_ptr(), batch, C.byref(want),
                                       grad.ctypes.data_as(C.POINTER(C.c_float))), "grad")
    assert got.value == want.value  # the same samples in the same order through the same kernels
