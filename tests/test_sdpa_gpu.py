"""Fused attention forward (ttlh_sdpa_fwd) against the float64 CPU reference
softmax(Q K^T s) V (oracle.tile_ops.sdpa_ref).

Bar (north star: bf16 out within a stated tolerance of an fp32 reference):
max |O - ref| <= 1e-2 * max |ref| and mean |O - ref| <= 4e-3 * mean |ref|
(bf16 rounding of P and of O contribute about 1e-3 each),
plus invariants that catch layout / indexing slips exactly: V = 1 gives
O = 1 (rows of P sum to one), a one-hot V column selects that column of P.
Sequence lengths that are multiples of 32 but not of 128 (a masked tail)
run with a guard region after the output.
"""

import math

import pytest
import torch

from oracle import tile_ops as O
from ttlhip import _lib as L

pytestmark = pytest.mark.gpu


def _run(q, k, v, scale, causal=False):
    from ttlhip import kernels as K
    out = torch.empty_like(q, device="cuda")
    K.sdpa_fwd(q.cuda(), k.cuda(), v.cuda(), out, scale, causal)
    torch.cuda.synchronize()
    return out.cpu()


# ttlh_sdpa_fwd_form: one or two groups of four waves (sdpa_fwd_kernel), eight
# waves (sdpa_w8_kernel).  A test that is there for one of them asks, so that a
# change of the choice cannot take its subject from it unseen.
ONE_GROUP, TWO_GROUPS, EIGHT_WAVES = 1, 2, 8


def _form(B, H, S, D=128, causal=False):
    return L.load().ttlh_sdpa_fwd_form(B, H, S, D, int(causal))


def _qkv(B, H, S, D, seed):
    return [O.seeded((B, H, S, D), "normal", seed + i) for i in range(3)]


def _check(out, ref):
    err = (out.double() - ref).abs()
    assert float(err.max()) <= 1e-2 * float(ref.abs().max()), float(err.max())
    assert float(err.mean()) <= 4e-3 * float(ref.abs().mean()), float(err.mean())


@pytest.mark.parametrize("B,H,S,D", [(1, 1, 128, 128), (2, 3, 256, 128), (1, 2, 384, 64),
                                    (1, 2, 768, 128)])
def test_sdpa_matches_reference(B, H, S, D):
    # few heads: sdpa_fwd_kernel whatever S is
    q, k, v = _qkv(B, H, S, D, 1)
    scale = 1.0 / math.sqrt(D)
    _check(_run(q, k, v, scale), O.sdpa_ref(q, k, v, scale))


@pytest.mark.parametrize("S", [128, 512])
def test_sdpa_causal(S):
    q, k, v = _qkv(1, 2, S, 128, 5)
    scale = 1.0 / math.sqrt(128)
    _check(_run(q, k, v, scale, causal=True), O.sdpa_ref(q, k, v, scale, causal=True))


def test_sdpa_rows_of_p_sum_to_one():
    q, k, _ = _qkv(1, 1, 256, 128, 9)
    v = torch.ones(1, 1, 256, 128, dtype=torch.bfloat16)
    out = _run(q, k, v, 1.0 / math.sqrt(128))
    assert float((out.float() - 1.0).abs().max()) <= 2 ** -7


def test_sdpa_one_hot_value_selects_probabilities():
    S = 256
    q, k, _ = _qkv(1, 1, S, 128, 11)
    v = torch.zeros(1, 1, S, 128, dtype=torch.bfloat16)
    v[0, 0, torch.arange(128), torch.arange(128)] = 1.0  # O[:, j] = P[:, j] for j < 128
    scale = 1.0 / math.sqrt(128)
    out = _run(q, k, v, scale)
    s = (q[0, 0].double() @ k[0, 0].double().T) * scale
    p = torch.softmax(s, -1)
    err = (out[0, 0].double() - p[:, :128]).abs()
    assert float(err.max()) <= 1e-2 * float(p.max())


def test_sdpa_config5_sampled_heads():
    B, H, S, D = 4, 32, 4096, 128
    assert _form(B, H, S) == EIGHT_WAVES
    q, k, v = _qkv(B, H, S, D, 21)
    scale = 1.0 / math.sqrt(D)
    out = _run(q, k, v, scale)
    for b, h in ((0, 0), (3, 31), (2, 17)):
        ref = O.sdpa_ref(q[b:b + 1, h:h + 1], k[b:b + 1, h:h + 1], v[b:b + 1, h:h + 1], scale)
        _check(out[b:b + 1, h:h + 1], ref)


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("scale", [-0.09, 0.0])
@pytest.mark.parametrize("causal", [False, True])
def test_sdpa_negative_and_zero_scale(scale, causal, D):
    # a negative scale flips which raw score is the row maximum; scale 0 is
    # uniform attention (plain / prefix mean of V)
    q, k, v = _qkv(1, 2, 256, D, 31)
    out = _run(q, k, v, scale, causal=causal)
    _check(out, O.sdpa_ref(q, k, v, scale, causal=causal))
    if scale == 0.0:
        vd = v.double()
        mean = (vd.cumsum(2) / torch.arange(1, 257, dtype=torch.float64).view(1, 1, -1, 1)
                if causal else vd.mean(2, keepdim=True).expand_as(vd))
        assert float((out.double() - mean).abs().max()) <= 1e-2 * float(mean.abs().max())


@pytest.mark.parametrize("B,H,S", [(1, 3, 1024), (3, 1, 512)])
def test_sdpa_several_query_blocks(B, H, S):
    # several query blocks per head and several cycles through the KV buffers; V = 1
    # in the second head (or batch) pins the row sums exactly
    q, k, v = _qkv(B, H, S, 128, 61)
    v[-1, -1] = 1.0
    scale = 1.0 / math.sqrt(128)
    out = _run(q, k, v, scale)
    ref = O.sdpa_ref(q, k, v, scale)
    rest = (slice(0, B - 1),) if B > 1 else (slice(None), slice(0, H - 1))
    _check(out[rest], ref[rest])
    assert float((out[-1, -1].float() - 1.0).abs().max()) <= 2 ** -7


def test_sdpa_causal_d64_and_value_layout():
    # D = 64 path, causal; V = column index pattern makes O's d layout exact:
    # every row of P sums to one, so O[:, :, :, d] == d (to bf16 rounding)
    q, k, _ = _qkv(1, 1, 384, 64, 41)
    v = torch.arange(64, dtype=torch.float32).repeat(1, 1, 384, 1).bfloat16()
    out = _run(q, k, v, 0.125, causal=True)
    expect = torch.arange(64, dtype=torch.float64).expand(1, 1, 384, 64)
    assert float((out.double() - expect).abs().max()) <= 63 * 2 ** -7


def test_sdpa_blocks_uneven_over_the_workgroups():
    # 75 heads x 4 query blocks = 300 blocks over at most one workgroup per
    # CU: workgroups walk one or two blocks (the eight-wave kernel's
    # persistent grid); sampled heads of every part of the sequence
    B, H, S, D = 1, 75, 1024, 128
    assert _form(B, H, S) == EIGHT_WAVES
    q, k, v = _qkv(B, H, S, D, 71)
    scale = 1.0 / math.sqrt(D)
    out = _run(q, k, v, scale)
    for h in (0, 37, 63, 64, 74):
        sl = (slice(None), slice(h, h + 1))
        _check(out[sl], O.sdpa_ref(q[sl], k[sl], v[sl], scale))


@pytest.mark.parametrize("B,H,S,seed", [(1, 4, 1024, 3), (1, 4, 1024, 4), (1, 2, 256, 5),
                                        (1, 34, 1024, 6), (2, 17, 1024, 7), (1, 130, 256, 8),
                                        (1, 70, 1024, 9)])
def test_sdpa_last_blocks_with_slow_kv_loads(B, H, S, seed):
    # K and V in pinned host memory: every K / V load crosses PCIe and takes
    # far longer than a step.  From 17 heads on the eight-wave kernel: every
    # workgroup's last query block (its only one, or with 70 heads its second)
    # stages no Q for a next block, and its end-of-step wait must still cover the
    # previous step's K / V loads, whose first fragments the next step prefetches.
    # A wait that counted the skipped Q loads reads stale fragments (max error
    # 0.28-0.59 of the output's range at [1, 4, 1024, 128] when that ran there),
    # now and then with device memory too.
    D = 128
    assert _form(B, H, S) == (EIGHT_WAVES if H >= 17 else TWO_GROUPS)
    g = torch.Generator().manual_seed(seed)
    q, k, v = (torch.randn(B, H, S, D, generator=g).bfloat16() for _ in range(3))
    kh, vh = k.pin_memory(), v.pin_memory()
    qd = q.cuda()
    out = torch.zeros_like(qd)
    L.call("ttlh_sdpa_fwd", qd.data_ptr(), kh.data_ptr(), vh.data_ptr(), out.data_ptr(), B, H, S,
           D, 0.1, 0, L.stream_ptr())
    torch.cuda.synchronize()
    out = out.cpu()
    for h in range(0, H, 1 if H < 10 else 7):
        sl = (slice(None), slice(h, h + 1))
        _check(out[sl], O.sdpa_ref(q[sl], k[sl], v[sl], 0.1))


@pytest.mark.parametrize("H,S", [(130, 256), (43, 768), (33, 1024)])
@pytest.mark.parametrize("scale", [0.09, -0.09, 0.0])
def test_sdpa_eight_waves(H, S, scale):
    # the eight-wave kernel with the fewest steps of a block (8, no pass of its
    # inner loop), one query block a workgroup and two; V = 1 in head 1 pins the row
    # sums, a one-hot V in head 2 shows the probabilities themselves
    print(f"sdpa eight waves {H}x{S} scale {scale}", flush=True)
    assert _form(1, H, S) == EIGHT_WAVES
    q, k, v = _qkv(1, H, S, 128, 91)
    v[0, 1] = 1.0
    v[0, 2] = 0.0
    v[0, 2, torch.arange(128), torch.arange(128)] = 1.0
    out = _run(q, k, v, scale)
    assert float((out[0, 1].float() - 1.0).abs().max()) <= 2 ** -7
    p = torch.softmax((q[0, 2].double() @ k[0, 2].double().T) * scale, -1)
    assert float((out[0, 2].double() - p[:, :128]).abs().max()) <= 1e-2 * float(p.max())
    for h in (0, 3, H // 2, H - 1):
        sl = (slice(None), slice(h, h + 1))
        _check(out[sl], O.sdpa_ref(q[sl], k[sl], v[sl], scale))


@pytest.mark.parametrize("jump", [False, True])
def test_sdpa_running_max_growth(jump):
    # scores that grow along kv (several rescales of O and l by the running
    # max) and, with jump, one late key whose score dwarfs every earlier one
    # (the rescale factor underflows to zero): the float64 softmax decides
    S, D = 512, 128
    q = torch.zeros(1, 2, S, D)
    q[..., 0] = 1.0
    q[..., 1] = torch.linspace(-1, 1, S)
    k = torch.zeros(1, 2, S, D)
    k[..., 0] = torch.linspace(0, 30, S)
    k[..., 1] = 0.5
    if jump:
        k[0, :, S - 70, 0] = 1000.0
    v = O.seeded((1, 2, S, D), "normal", 51)
    q, k = q.bfloat16(), k.bfloat16()
    for causal in (False, True):
        out = _run(q, k, v, 1.0, causal=causal)
        _check(out, O.sdpa_ref(q, k, v, 1.0, causal=causal))


def test_sdpa_running_max_growth_in_later_blocks_of_a_workgroup():
    # 260 heads x 2 query blocks = 520 blocks over at most one workgroup per
    # CU: workgroups walk 2 or 3 blocks, and the running-max rescales (scores
    # growing along kv, one late key far above the rest) happen in every block,
    # so a block's rescale state must not leak into the next
    B, H, S, D = 1, 260, 512, 128
    assert _form(B, H, S) == EIGHT_WAVES
    q = torch.zeros(B, H, S, D)
    q[..., 0] = 1.0
    q[..., 1] = torch.linspace(-1, 1, S)
    k = torch.zeros(B, H, S, D)
    k[..., 0] = torch.linspace(0, 30, S)
    k[..., 1] = 0.5
    k[:, 1::2, S - 70, 0] = 1000.0
    v = O.seeded((B, H, S, D), "normal", 81)
    q, k = q.bfloat16(), k.bfloat16()
    out = _run(q, k, v, 1.0)
    for h in (0, 1, 127, 200, 258, 259):
        sl = (slice(None), slice(h, h + 1))
        _check(out[sl], O.sdpa_ref(q[sl], k[sl], v[sl], 1.0))


@pytest.mark.parametrize("S", [32, 96, 160, 224, 416])
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("causal", [False, True])
def test_sdpa_ragged_seq(S, D, causal):
    # S a multiple of 32 but not of 128: the last query block holds waves past
    # the sequence and the last KV block rows past it (masked, read as zero).
    # The output sits in a larger buffer whose tail must stay untouched.
    B, H = 1, 3
    q, k, v = _qkv(B, H, S, D, S + D)
    scale = 1.0 / math.sqrt(D)
    from ttlhip import kernels as K
    n = B * H * S * D
    big = torch.full((n + 64 * D,), 3.0, dtype=torch.bfloat16, device="cuda")
    out = big[:n].view(B, H, S, D)
    K.sdpa_fwd(q.cuda(), k.cuda(), v.cuda(), out, scale, causal)
    torch.cuda.synchronize()
    _check(out.cpu(), O.sdpa_ref(q, k, v, scale, causal=causal))
    assert bool((big[n:] == 3.0).all()), "write past the output"
    ones = torch.ones_like(v)
    out1 = _run(q, k, ones, scale, causal=causal)
    assert float((out1.float() - 1.0).abs().max()) <= 2 ** -7


@pytest.mark.parametrize("scale", [-0.11, 0.0])
def test_sdpa_ragged_negative_and_zero_scale(scale):
    q, k, v = _qkv(1, 2, 96, 128, 77)
    _check(_run(q, k, v, scale), O.sdpa_ref(q, k, v, scale))


@pytest.mark.parametrize("S,D,causal", [(384, 128, False), (256, 64, False), (96, 128, False),
                                        (512, 128, True), (256, 64, True)])
def test_sdpa_other_kernels_with_slow_loads(S, D, causal):
    # sdpa_fwd_kernel (one and two groups, whole and ragged, with and without
    # the mask) with Q, K and V in pinned host memory: loads far slower than any
    # step of its pipeline
    assert _form(1, 2, S, D, causal) == (TWO_GROUPS if S > 192 else ONE_GROUP)
    g = torch.Generator().manual_seed(S + D)
    q, k, v = (torch.randn(1, 2, S, D, generator=g).bfloat16() for _ in range(3))
    qh, kh, vh = q.pin_memory(), k.pin_memory(), v.pin_memory()
    out = torch.zeros(1, 2, S, D, dtype=torch.bfloat16, device="cuda")
    L.call("ttlh_sdpa_fwd", qh.data_ptr(), kh.data_ptr(), vh.data_ptr(), out.data_ptr(), 1, 2, S,
           D, 0.1, int(causal), L.stream_ptr())
    torch.cuda.synchronize()
    _check(out.cpu(), O.sdpa_ref(q, k, v, 0.1, causal))


@pytest.mark.parametrize("B,H,S,D,causal", [(1, 2, 160, 128, True), (1, 2, 192, 64, False),
                                            (1, 1, 1056, 128, True), (2, 16, 1024, 64, True),
                                            (1, 32, 1120, 128, True), (1, 65, 544, 64, False),
                                            (3, 24, 480, 128, True)])
def test_sdpa_block_forms(B, H, S, D, causal):
    # sdpa_fwd_kernel's forms (one and two groups of waves, whole and ragged
    # sequences) and the causal block order: 3 to 33 KV blocks, so the groups'
    # shares are equal and unequal, heads that an XCD's share divides and not
    print(f"sdpa forms {B}x{H}x{S}x{D} causal={causal}", flush=True)
    q, k, v = _qkv(B, H, S, D, 41)
    _check(_run(q, k, v, 1.0 / math.sqrt(D), causal=causal),
           O.sdpa_ref(q, k, v, 1.0 / math.sqrt(D), causal=causal))


@pytest.mark.parametrize("S", [256, 2048])
def test_sdpa_scores_of_minus_infinity(S):
    # keys whose scores are -inf drop out, a whole KV block of them too
    # (the first one, and in the second group's share)
    g = torch.Generator().manual_seed(5)
    q = torch.rand(1, 2, S, 128, generator=g).bfloat16() + 0.5  # positive
    k, v = (torch.randn(1, 2, S, 128, generator=g).bfloat16() for _ in range(2))
    k[:, :, :128, 3] = -float("inf")
    k[:, :, 200:230, 3] = -float("inf")
    got = _run(q, k, v, 0.09)
    keep = torch.isfinite(k[0, 0, :, 3])
    ref = O.sdpa_ref(q, k[:, :, keep], v[:, :, keep], 0.09)
    _check(got, ref)


@pytest.mark.parametrize("H,S", [(3, 256), (3, 2048), (17, 2048), (130, 256)])
def test_sdpa_leading_scores_of_minus_infinity(H, S):
    # with few blocks sdpa_fwd_kernel, with more than 256 sdpa_w8_kernel.  Even
    # queries score -inf on the first keys (-3e38 times 64), odd ones do not see
    # that column; every finite score is near -270, far below where exp underflows
    # next to a maximum that would have stayed at 0.  Head 1 has three keys left, all
    # at the end, and head 2 none: its even rows are 0 / 0.
    print(f"sdpa -inf {H}x{S}", flush=True)
    assert _form(1, H, S) == (TWO_GROUPS if H == 3 else EIGHT_WAVES)
    q, k, v = _qkv(1, H, S, 128, 23)
    q[..., 3] = 0.0
    q[:, :, ::2, 3] = 64.0
    q[..., 5], k[..., 5] = 1.0, -3008.0
    k[..., 3] = 0.0
    k[:, :, :40, 3] = k[:, :, 64:160, 3] = -3e38
    k[:, 1, :S - 3, 3] = -3e38
    k[:, 2, :, 3] = -3e38
    got = _run(q, k, v, 0.09)
    for h in (0, 1, 2, H - 1):
        keep = k[0, h, :, 3] == 0
        even, odd = q[:, h:h + 1, ::2].clone(), q[:, h:h + 1, 1::2]
        _check(got[:, h:h + 1, 1::2], O.sdpa_ref(odd, k[:, h:h + 1], v[:, h:h + 1], 0.09))
        if bool(keep.any()):
            _check(got[:, h:h + 1, ::2],
                   O.sdpa_ref(even, k[:, h:h + 1, keep], v[:, h:h + 1, keep], 0.09))
        else:
            assert bool(torch.isnan(got[:, h, ::2]).all())


@pytest.mark.parametrize("S", [96, 480])
@pytest.mark.parametrize("D", [64, 128])
def test_sdpa_infinite_value_in_a_ragged_last_row(S, D):
    # the rows past the sequence are zeros, not copies of its last one: that
    # row's infinity reaches its column once, and never as 0 * inf
    q, k, v = _qkv(1, 2, S, D, 19)
    ref = O.sdpa_ref(q, k, v, 0.09)
    v[:, :, S - 1, 5] = float("inf")
    got = _run(q, k, v, 0.09)
    assert bool((got[..., 5] == float("inf")).all())
    rest = [d for d in range(D) if d != 5]
    _check(got[..., rest], ref[..., rest])


@pytest.mark.parametrize("S,D,causal", [(224, 128, True), (416, 64, False), (160, 64, True),
                                        (480, 128, False)])
def test_sdpa_ragged_forms_with_slow_loads(S, D, causal):
    # one and two groups, the last block half past the sequence: its zeros are
    # written after its loads have landed, however late those are
    test_sdpa_other_kernels_with_slow_loads(S, D, causal)
