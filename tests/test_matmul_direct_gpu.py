"""The register-direct GEMM kernels on the MI355X at the edges of their blocks:
one tile of rows, columns that end inside a block, K shorter than the waves'
stages, K divided among workgroups (scratch), outputs without vector
alignment.  The reference is the float64 product of the same inputs.  Bounds
as for the other GEMM kernels: fp32 sums of K products (1e-6 sqrt(K) of the
largest result) and, for bf16 results, one rounding (2^-8 of the value)."""

import math
import threading

import pytest
import torch

from oracle import bfp8 as OB
from oracle import tile_ops as O
from ttlhip import _lib as L
from ttlhip import expr as X
from ttlhip import kernels as Kn

pytestmark = pytest.mark.gpu

# (M, K, N): every block shape, whole and cut; K of one stage, of fewer stages
# than waves, and long enough to be divided
SHAPES = [(32, 32, 32), (32, 96, 96), (64, 4096, 96), (96, 2048, 160), (32, 11008, 288),
          (160, 1024, 1056), (224, 544, 1504), (544, 288, 2080), (1056, 160, 3104),
          (2080, 96, 2016)]


def _check(got, a, b, bf16_out):
    exact = a.cpu().double() @ b.cpu().double()
    bound = 1e-6 * math.sqrt(a.shape[1]) * float(exact.abs().max())
    if bf16_out:
        bound = bound + exact.abs() * 2.0 ** -8
    err = (got.cpu().double() - exact).abs()
    assert bool((err <= bound).all()), float(err.max())


def _operands(M, K, N, seed, dtype=torch.bfloat16):
    std = K ** -0.25
    return (O.seeded((M, K), "normal", seed, dtype, std=std).cuda(),
            O.seeded((K, N), "normal", seed + 1, dtype, std=std).cuda())


@pytest.mark.parametrize("M,K,N", SHAPES)
def test_bf16_blocks(M, K, N):
    print(f"direct bf16 {M}x{K}x{N}", flush=True)
    a, b = _operands(M, K, N, 3)
    # a guard column on each side: results outside the block stay untouched,
    # and the odd pitch takes the stores without vector alignment
    buf = torch.full((M, N + 3), 7.0, dtype=torch.bfloat16, device="cuda")
    Kn.matmul(a, b, buf[:, 1:N + 1])
    wide = torch.empty(M, N, dtype=torch.bfloat16, device="cuda")
    for _ in range(3):  # the counters of the divided products reset themselves
        wide.zero_()
        Kn.matmul(a, b, wide)
        _check(wide, a, b, True)
    assert torch.equal(buf[:, 1:N + 1], wide)
    assert bool((buf[:, 0] == 7).all()) and bool((buf[:, N + 1:] == 7).all())


@pytest.mark.parametrize("K", [32, 64, 96, 128, 160, 192, 224, 256, 352])
def test_bf16_blocks_of_128(K):
    # mm_mid_kernel: every number of stages around its ring of four buffers,
    # blocks cut in both directions, accumulation and fp32 results
    M, N = 2080, 1952
    print(f"mid bf16 K={K}", flush=True)
    a, b = _operands(M, K, N, 11)
    c = torch.full((M, N + 2), 7.0, dtype=torch.bfloat16, device="cuda")
    Kn.matmul(a, b, c[:, :N])
    _check(c[:, :N], a, b, True)
    assert bool((c[:, N:] == 7).all())
    odd = torch.full((M, N + 3), 7.0, dtype=torch.bfloat16, device="cuda")
    Kn.matmul(a, b, odd[:, 1:N + 1])
    assert torch.equal(odd[:, 1:N + 1], c[:, :N])
    assert bool((odd[:, 0] == 7).all()) and bool((odd[:, N + 1:] == 7).all())
    f = O.seeded((M, N), "normal", 12, torch.float32).cuda()
    f0 = f.clone()
    Kn.matmul(a, b, f, accumulate=True)
    _check(f - f0, a, b, False)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("M,K,N", [(3328, 1024, 3072), (4064, 512, 4064)])
def test_blocks_of_256_into_a_result_off_its_pairs(M, K, N, dtype):
    # mm_dma_kernel (below and above 192 blocks, whole and cut) writes two columns at
    # once, also where a column slice or an odd pitch leaves them unaligned
    print(f"unaligned pairs {M}x{K}x{N} {dtype}", flush=True)
    a, b = _operands(M, K, N, 29)
    c = torch.empty(M, N, dtype=dtype, device="cuda")
    Kn.matmul(a, b, c)
    _check(c, a, b, dtype == torch.bfloat16)
    odd = torch.full((M, N + 3), 7.0, dtype=dtype, device="cuda")
    Kn.matmul(a, b, odd[:, 1:N + 1])
    assert torch.equal(odd[:, 1:N + 1], c)
    assert bool((odd[:, 0] == 7).all()) and bool((odd[:, N + 1:] == 7).all())
    c0 = O.seeded((M, N), "normal", 30, dtype).cuda()
    wide = c0.clone()
    Kn.matmul(a, b, wide, accumulate=True)
    odd[:, 1:N + 1] = c0
    Kn.matmul(a, b, odd[:, 1:N + 1], accumulate=True)
    assert torch.equal(odd[:, 1:N + 1], wide)
    assert bool((odd[:, 0] == 7).all()) and bool((odd[:, N + 1:] == 7).all())


@pytest.mark.parametrize("M,K,N,pitch", [(4096, 96, 3072, 2 ** 19 + 8), (4096, 32, 3104, 2 ** 19 + 5),
                                        (32, 2048, 96, 2 ** 26 + 1)])
def test_bf16_results_past_32_bit_offsets(M, K, N, pitch):
    # the result spans 2^31 elements and more: mm_bf16_kernel in place of the kernels
    # with 32-bit offsets of C (192 blocks of 256x256 and more), and the
    # register-direct kernels, whose offsets have 64
    print(f"far results {M}x{K}x{N} pitch {pitch}", flush=True)
    a, b = _operands(M, K, N, 37)
    buf = torch.full(((M - 1) * pitch + N + 2,), 7.0, dtype=torch.bfloat16, device="cuda")
    c = buf[1:].as_strided((M, N), (pitch, 1), 1)
    Kn.matmul(a, b, c)
    _check(c, a, b, True)
    c0 = O.seeded((M, N), "normal", 38, torch.bfloat16).cuda()
    c.copy_(c0)
    Kn.matmul(a, b, c, accumulate=True)
    exact = a.cpu().double() @ b.cpu().double() + c0.cpu().double()
    bound = 1e-6 * math.sqrt(K) * float(exact.abs().max()) + exact.abs() * 2.0 ** -8
    assert bool(((c.cpu().double() - exact).abs() <= bound).all())
    around = buf.as_strided((M, N + 2), (pitch, 1), 0)
    assert bool((around[:, 0] == 7).all()) and bool((around[:, N + 1] == 7).all())


@pytest.mark.parametrize("M,K,N", [(4096, 32, 3072), (4096, 96, 3104), (32, 64, 49152)])
def test_sums_in_the_fused_epilogues_order(M, K, N):
    # problems that the fused epilogue takes give the same bits with and
    # without it, whichever kernel runs the plain product
    a, b = _operands(M, K, N, 19)
    c = torch.zeros(M, N, dtype=torch.bfloat16, device="cuda")
    Kn.matmul(a, b, c)
    leaf = X.Leaf(0, torch.bfloat16)
    prog = X.compile_expr(X.Unary("relu", leaf, torch.bfloat16))
    d = torch.zeros_like(c)
    Kn.matmul_eltwise(a, b, prog, [None] * len(prog.steps), 0, d, (0, 0, M, N))
    assert torch.equal(d, torch.relu(c))


def test_bf16_blocks_of_128_with_slow_operand_loads():
    # A and B in pinned host memory: every stage's loads take far longer than
    # a stage, so a wait that covered too few of them would read a stale stage
    a, b = _operands(2080, 352, 1952, 17)
    pa, pb = a.cpu().pin_memory(), b.cpu().pin_memory()
    c = torch.zeros(2080, 1952, dtype=torch.bfloat16, device="cuda")
    L.call("ttlh_matmul", pa.data_ptr(), L.TTLH_BF16, 352, pb.data_ptr(), L.TTLH_BF16, 1952,
           c.data_ptr(), L.TTLH_BF16, 1952, 2080, 1952, 352, 0, L.stream_ptr())
    torch.cuda.synchronize()
    _check(c, a, b, True)


@pytest.mark.parametrize("M,K,N", [(32, 32, 32), (64, 2048, 96), (96, 160, 224), (32, 4096, 32),
                                   (544, 96, 608), (1056, 64, 1504), (1760, 96, 1792)])
def test_f32_blocks(M, K, N):
    print(f"direct f32 {M}x{K}x{N}", flush=True)
    a, b = _operands(M, K, N, 13, torch.float32)
    buf = torch.full((M, N + 3), 7.0, device="cuda")
    Kn.matmul(a, b, buf[:, 1:N + 1])
    wide = torch.zeros(M, N, device="cuda")
    for _ in range(2):
        Kn.matmul(a, b, wide)
        _check(wide, a, b, False)
    assert torch.equal(buf[:, 1:N + 1], wide)
    assert bool((buf[:, 0] == 7).all()) and bool((buf[:, N + 1:] == 7).all())
    Kn.matmul(a, b, wide, accumulate=True)
    torch.testing.assert_close(wide, 2 * buf[:, 1:N + 1], rtol=1e-6, atol=1e-6)
    # operands off the vector alignment take the kernel through LDS
    oa, ob = torch.empty(M, K + 1, device="cuda"), torch.empty(K, N + 1, device="cuda")
    oa[:, 1:], ob[:, 1:] = a, b
    Kn.matmul(oa[:, 1:], ob[:, 1:], wide)
    _check(wide, a, b, False)


@pytest.mark.parametrize("M,K,N", [(32, 4096, 96), (96, 288, 1056)])
def test_bf16_accumulate_f32(M, K, N):
    a, b = _operands(M, K, N, 5)
    c0 = O.seeded((M, N), "normal", 7, torch.float32).cuda()
    c = c0.clone()
    Kn.matmul(a, b, c, accumulate=True)
    _check(c - c0, a, b, False)


def test_divided_product_under_capture_and_on_two_streams():
    # under capture one workgroup takes all parts of K (a replay may run beside
    # launches that use the scratch); two streams have a scratch each
    a, b = _operands(32, 4096, 256, 9)
    c = torch.zeros(32, 256, dtype=torch.bfloat16, device="cuda")
    Kn.matmul(a, b, c)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    d = torch.zeros_like(c)
    with torch.cuda.graph(g):
        Kn.matmul(a, b, d)
    for _ in range(3):
        d.zero_()
        g.replay()
        Kn.matmul(a, b, c)
        torch.cuda.synchronize()
        _check(d, a, b, True)
        _check(c, a, b, True)
    streams = [torch.cuda.Stream() for _ in range(2)]
    outs = [[torch.zeros_like(c) for _ in range(8)] for _ in streams]
    torch.cuda.synchronize()
    for i in range(8):
        for s, o in zip(streams, outs):
            Kn.matmul(a, b, o[i], stream=s)
    torch.cuda.synchronize()
    for o in outs:
        assert all(torch.equal(x, c) for x in o)
    Kn.release_workspaces()
    Kn.matmul(a, b, c)
    _check(c, a, b, True)


def test_scratch_of_a_stream_while_another_thread_captures():
    # the first product of a stream takes its scratch; that allocation ends
    # neither in an error nor with the other thread's (global mode) capture
    a, b = _operands(32, 4096, 256, 11)
    c, d = (torch.zeros(32, 256, dtype=torch.bfloat16, device="cuda") for _ in range(2))
    Kn.matmul(a, b, c)
    Kn.release_workspaces()
    side, errors = torch.cuda.Stream(), []

    def first_product():
        try:
            Kn.matmul(a, b, c, stream=side)
        except Exception as e:  # reported by the main thread
            errors.append(e)

    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        Kn.matmul(a, b, d)
        t = threading.Thread(target=first_product)
        t.start()
        t.join()
    assert not errors, errors
    g.replay()
    torch.cuda.synchronize()
    _check(c, a, b, True)
    _check(d, a, b, True)


def test_scratches_are_bounded(monkeypatch):
    monkeypatch.setattr(Kn, "_MATMUL_SCRATCH_MAX", 2)
    Kn.release_workspaces()
    a, b = _operands(32, 4096, 256, 13)
    outs = [torch.zeros(32, 256, dtype=torch.bfloat16, device="cuda") for _ in range(4)]
    streams = [torch.cuda.Stream() for _ in outs]
    torch.cuda.synchronize()
    for _ in range(3):
        for s, o in zip(streams, outs):
            Kn.matmul(a, b, o, stream=s)
            assert len(Kn._MATMUL_SCRATCH) <= 2
    torch.cuda.synchronize()
    for o in outs:
        _check(o, a, b, True)


def test_scratch_only_where_k_may_be_divided(monkeypatch):
    # large products, short sums and packed weights' two passes take none; without
    # memory for one the product runs all the same, with the same bits
    Kn.release_workspaces()
    for M, K, N, dt in [(1024, 4096, 1024, torch.bfloat16), (32, 1024, 256, torch.bfloat16),
                        (512, 2048, 512, torch.float32)]:
        a, b = _operands(M, K, N, 45, dt)
        Kn.matmul(a, b, torch.zeros(M, N, dtype=dt, device="cuda"))
        assert not Kn._MATMUL_SCRATCH
    a, b = _operands(32, 4096, 256, 46)
    c, d = (torch.zeros(32, 256, dtype=torch.bfloat16, device="cuda") for _ in range(2))

    def no_memory(*args, **kwargs):
        raise torch.OutOfMemoryError("no memory for the scratch")

    with monkeypatch.context() as m:
        m.setattr(Kn.torch, "zeros", no_memory)
        Kn.matmul(a, b, c)
    assert not Kn._MATMUL_SCRATCH
    Kn.matmul(a, b, d)
    assert len(Kn._MATMUL_SCRATCH) == 1
    assert torch.equal(c, d)
    _check(d, a, b, True)


def _packed(w, bits):
    return OB.pack_c(w) if bits == 8 else OB.pack4_c(w)


def _unpacked(q, K, N, bits):
    return OB.unpack_c(q, K, N) if bits == 8 else OB.unpack4_c(q, K, N)


def _matmul_packed(a, q, c, bits):
    if bits == 8:
        Kn.matmul_bfp8w(a, q, c, two_pass=False)
    else:
        Kn.matmul_bfp4w(a, q, c)


@pytest.mark.parametrize("bits", [8, 4])
@pytest.mark.parametrize("M,K,N", [s for s in SHAPES if s[0] < 512] + [(480, 160, 1504)])
def test_packed_weights(M, K, N, bits):
    print(f"direct packed {bits} {M}x{K}x{N}", flush=True)
    a = O.seeded((M, K), "normal", 21, torch.bfloat16, std=K ** -0.5).cuda()
    q = _packed(O.seeded((K, N), "normal", 22, torch.float32), bits)
    w = _unpacked(q, K, N, bits)
    qd = q.cuda()
    c = torch.empty(M, N, dtype=torch.bfloat16, device="cuda")
    for _ in range(2):
        c.zero_()
        _matmul_packed(a, qd, c, bits)
        _check(c, a, w, True)
    off = torch.empty(q.numel() + 8, dtype=torch.uint8, device="cuda")[8:]
    off.copy_(qd)  # tiles on 8 bytes, not 16
    d = torch.empty_like(c)
    _matmul_packed(a, off, d, bits)
    assert torch.equal(c, d)


@pytest.mark.parametrize("bits", [8, 4])
@pytest.mark.parametrize("K", [96, 352])
def test_packed_decode_is_exact(K, bits):
    # rows of the identity read the weights themselves: random bytes with every
    # finite exponent, subnormal results among them
    N, per = 160, 1088 if bits == 8 else 576
    g = torch.Generator().manual_seed(31)
    q = torch.randint(0, 256, ((K // 32) * (N // 32), per), generator=g, dtype=torch.uint8)
    q[:, :64] = torch.randint(0, 255, (q.shape[0], 64), generator=g, dtype=torch.uint8)
    q = q.flatten()
    c = torch.empty(K, N, dtype=torch.bfloat16, device="cuda")
    _matmul_packed(torch.eye(K, dtype=torch.bfloat16, device="cuda"), q.cuda(), c, bits)
    w = _unpacked(q, K, N, bits)
    assert torch.equal(c.cpu().float(), w.float())


@pytest.mark.parametrize("K,N", [(128, 3072), (96, 3104)])
def test_packed_weights_in_blocks_of_256_into_a_result_off_its_pairs(K, N):
    # mm_dq_kernel and mm256_kernel, as above
    M = 4096
    print(f"unaligned pairs packed {M}x{K}x{N}", flush=True)
    a = O.seeded((M, K), "normal", 33, torch.bfloat16, std=K ** -0.5).cuda()
    q = OB.pack_c(O.seeded((K, N), "normal", 34, torch.float32))
    qd = q.cuda()
    c = torch.empty(M, N, dtype=torch.bfloat16, device="cuda")
    _matmul_packed(a, qd, c, 8)
    _check(c, a, OB.unpack_c(q, K, N), True)
    odd = torch.full((M, N + 3), 7.0, dtype=torch.bfloat16, device="cuda")
    _matmul_packed(a, qd, odd[:, 1:N + 1], 8)
    assert torch.equal(odd[:, 1:N + 1], c)
    assert bool((odd[:, 0] == 7).all()) and bool((odd[:, N + 1:] == 7).all())


@pytest.mark.parametrize("bits", [8, 4])
@pytest.mark.parametrize("M", [32, 96])
def test_packed_weights_and_rows_far_apart(M, bits):
    # rows of A 2^24 elements apart: past the decoding kernels' 32-bit offsets, so
    # bfloat8_b goes to mm_bf16_kernel's decoding form, bfloat4_b to the two passes
    K, N, pitch = 160, 96, 2 ** 24
    print(f"packed {bits} pitch {pitch} M {M}", flush=True)
    buf = torch.empty((M - 1) * pitch + K, dtype=torch.bfloat16, device="cuda")
    a = buf.as_strided((M, K), (pitch, 1))
    a.copy_(O.seeded((M, K), "normal", 35, torch.bfloat16, std=K ** -0.5))
    q = _packed(O.seeded((K, N), "normal", 36, torch.float32), bits)
    c = torch.empty(M, N, dtype=torch.bfloat16, device="cuda")
    _matmul_packed(a, q.cuda(), c, bits)
    _check(c, a, _unpacked(q, K, N, bits), True)


@pytest.mark.parametrize("kind", [torch.bfloat16, torch.float32, 8, 4])
@pytest.mark.parametrize("M,K,N", [(32, 2048, 96), (32, 11008, 288), (64, 4096, 1504),
                                   (96, 4000, 3968), (160, 2080, 2080)])
def test_divided_products_bits_are_their_sizes(M, K, N, kind):
    # K in two and four parts of 32x64, 32x128 and (fp32) 32x32 blocks, and cut
    # blocks: the same bits with a workgroup for each part, under capture and without
    # a scratch at all
    print(f"parts {M}x{K}x{N} {kind}", flush=True)
    if kind in (8, 4):
        a = O.seeded((M, K), "normal", 41, torch.bfloat16, std=K ** -0.5).cuda()
        b = _packed(O.seeded((K, N), "normal", 42, torch.float32), kind).cuda()
        dt, code = torch.bfloat16, kind

        def run(out):
            _matmul_packed(a, b, out, kind)
    else:
        a, b = _operands(M, K, N, 41, kind)
        dt, code = kind, L.dtype_code(kind)

        def run(out):
            Kn.matmul(a, b, out)
    eager, captured, bare = (torch.zeros(M, N, dtype=dt, device="cuda") for _ in range(3))
    run(eager)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        run(captured)
    for _ in range(3):
        captured.zero_()
        g.replay()
        run(eager)
        torch.cuda.synchronize()
        assert torch.equal(captured, eager)
    L.call("ttlh_matmul_scratch", a.data_ptr(), L.dtype_code(a.dtype), K, b.data_ptr(), code, N,
           bare.data_ptr(), L.dtype_code(dt), N, M, N, K, 0, 0, 0, L.stream_ptr())
    assert torch.equal(bare, eager)
