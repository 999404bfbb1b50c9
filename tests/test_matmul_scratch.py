"""Which scratch a product's launch gets (ttlhip.kernels._matmul_scratch), without
a GPU: the cached tensors are stand-ins."""

from types import SimpleNamespace

import torch

from ttlhip import kernels as Kn


def _stream(index):
    return SimpleNamespace(device=torch.device("cuda", index), cuda_stream=0)


def test_a_scratch_is_its_own_devices(monkeypatch):
    # every device's default stream has handle 0: device 0's scratch is not for a
    # launch on device 1's stream, whatever device the tensors are on
    mine = object()
    monkeypatch.setattr(Kn, "_MATMUL_SCRATCH", {(0, 0): mine})
    d0, d1 = torch.device("cuda", 0), torch.device("cuda", 1)
    assert Kn._matmul_scratch(d0, _stream(0), 0) is mine
    assert Kn._matmul_scratch(d0, _stream(1), 0) is None
    assert Kn._matmul_scratch(d1, _stream(0), 0) is None
    for current, expect in ((0, mine), (1, None)):
        monkeypatch.setattr(torch._C, "_cuda_getDevice", lambda: current, raising=False)
        assert Kn._matmul_scratch(d0, None, 0) is expect
