"""Which products the row GEMMs take.  The rule is about sizes, types and
addresses, so it is checked here on stand-ins, without a GPU: whatever it takes
is read by kernels that know only x's sizes and the number of weight rows."""
from types import SimpleNamespace

import pytest
import torch

from agentfield_amd import ops


def mat(*shape, dtype=torch.bfloat16, device="cuda:0", contiguous=True,
        addr=1 << 20):
    return SimpleNamespace(
        shape=torch.Size(shape), dtype=dtype, device=torch.device(device),
        is_cuda=device.startswith("cuda"), is_contiguous=lambda: contiguous,
        data_ptr=lambda: addr, dim=lambda: len(shape))


@pytest.mark.parametrize("M", [1, 16, 17, 128])
@pytest.mark.parametrize("N,K", [(64, 64), (4096, 512), (128256, 4096)])
def test_taken(M, N, K):
    assert ops._rows_ok(mat(M, K), mat(N, K))


@pytest.mark.parametrize("x,w", [
    (mat(4, 512), mat(128, 448)),            # rows longer than the weights'
    (mat(4, 448), mat(128, 512)),            # and shorter
    (mat(512), mat(128, 512)),
    (mat(2, 4, 512), mat(128, 512)),
    (mat(4, 512), mat(2, 128, 512)),
    (mat(0, 512), mat(128, 512)),
    (mat(129, 512), mat(128, 512)),
    (mat(4, 0), mat(128, 0)),
    (mat(4, 512), mat(0, 512)),
    (mat(4, 512), mat(96, 512)),
    (mat(4, 480), mat(128, 480)),
    (mat(4, 512), mat(128, 512, device="cpu")),
    (mat(4, 512, device="cpu"), mat(128, 512)),
    (mat(4, 512), mat(128, 512, device="cuda:1")),
    (mat(4, 512, dtype=torch.float32), mat(128, 512, dtype=torch.float32)),
    (mat(4, 512), mat(128, 512, dtype=torch.float16)),
    (mat(4, 512, contiguous=False), mat(128, 512)),
    (mat(4, 512), mat(128, 512, contiguous=False)),
    (mat(4, 512, addr=8), mat(128, 512)),
    (mat(4, 512), mat(128, 512, addr=2)),
], ids=lambda t: f"{'x'.join(map(str, t.shape))}")
def test_left_to_the_library(x, w):
    assert not ops._rows_ok(x, w)
