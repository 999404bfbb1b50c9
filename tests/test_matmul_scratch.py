"""Which scratch a product's launch gets (ttlhip.kernels._matmul_scratch), without
a GPU: the cached tensors are stand-ins."""

from types import SimpleNamespace

import pytest
import torch

from ttlhip import _lib as L
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


@pytest.mark.parametrize("a,b,M,N,K,uses", [
    (L.TTLH_BF16, L.TTLH_BF16, 32, 4096, 11008, True),
    (L.TTLH_BF16, L.TTLH_BF16, 32, 16384, 2048, True),
    (L.TTLH_BF16, L.TTLH_BF16, 32, 4096, 2016, False),   # a wave would keep too little of K
    (L.TTLH_BF16, L.TTLH_BF16, 1024, 1024, 11008, False),
    (L.TTLH_F32, L.TTLH_F32, 256, 256, 512, True),
    (L.TTLH_F32, L.TTLH_F32, 2048, 2048, 2048, False),
    (L.TTLH_BF16, L.TTLH_BFP8, 32, 4096, 4096, True),
    (L.TTLH_BF16, L.TTLH_BFP4, 32, 11008, 4096, False),
    (L.TTLH_BF16, L.TTLH_BF16, 0, 32, 32, False)])
def test_which_products_ask_for_it(a, b, M, N, K, uses):
    need = L.load().ttlh_matmul_scratch_bytes(a, b, M, N, K)
    assert need == (L.MATMUL_SCRATCH_BYTES if uses else 0)
