"""Device memory after a training: the sample order of a large one is given back."""
import ctypes as C

import pytest
import torch

from cleo_amd import abi

pytestmark = pytest.mark.gpu


def test_large_training_gives_its_order_back(gpu):
    n = (1 << 24) + 3
    print(f"case: device memory after a training on {n} samples", flush=True)
    x = torch.zeros((n, 8), device="cuda", dtype=torch.float32)
    x[:, :6] = torch.rand((n, 6), device="cuda")
    y = torch.rand(n, device="cuda")
    torch.cuda.synchronize()
    d = abi.Domain(gpu, 64, (1, 1, 1), [0.0, 1.0], [0.0, 1.0], [0.0, 1.0])
    loss = C.c_float()

    def train(samples):
        tp = abi.MLPTrainParams(1, 65536, 1e-3, 0.9, 0.999, 1e-8, 5)
        d.check(gpu.lib.cleo_mlp_train(d.h, x.data_ptr(), y.data_ptr(), samples, C.byref(tp), C.byref(loss)), "train")
        return torch.cuda.mem_get_info()[0]

    small = train(65536)  # the buffers of a batch, and what the first launches take
    large = train(n)
    assert small - large < 10 * n  # the order's 20 bytes per sample are free again
    assert train(65536) > 0
