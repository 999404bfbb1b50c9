"""Column reductions of a plain bf16 operand (reduce_cols_strip_kernel) at the
edges of its strips of 64 columns, its passes of 64 rows and its row shares,
against float64: maxima exact, sums within the fp32 bound of their terms."""

import pytest
import torch

from oracle import tile_ops as O
from ttlhip import expr as X
from ttlhip import kernels as K

pytestmark = pytest.mark.gpu


def _run(x, kind, region, out, **kw):
    K.reduce(X.compile_expr(X.Leaf(0, x.dtype)), [K.OperandMap(x)], kind, [0], out, region, **kw)


def _check(got, part, kind, scale=1.0):
    v = part.cpu().double() * scale
    if kind == "max":
        assert torch.equal(got.cpu().double(), v.amax(0))
    else:
        bound = v.shape[0] * 2.0 ** -24 * v.abs().sum(0) + 1e-30
        assert bool(((got.cpu().double() - v.sum(0)).abs() <= bound).all())


@pytest.mark.parametrize("kind", ["sum", "max"])
@pytest.mark.parametrize("h,w", [(1, 8), (2, 64), (63, 72), (64, 200), (65, 4104), (513, 64),
                                 (1024, 96), (2047, 136), (2048, 64), (4099, 264), (9000, 24),
                                 (2056, 32768), (66000, 72), (1000000, 8)])
def test_strips(h, w, kind):
    print(f"column strips {h}x{w} {kind}", flush=True)
    x = O.seeded((h, w), "normal", 3).cuda()
    out = torch.full((1, w + 2), 7.0, device="cuda")
    _run(x, kind, (0, 0, h, w), out, out_origin=(0, 1), scale=0.5)
    _check(out[0, 1:w + 1], x, kind, 0.5)
    assert float(out[0, 0]) == 7 and float(out[0, w + 1]) == 7


@pytest.mark.parametrize("kind", ["sum", "max"])
def test_region_of_a_strided_operand_with_padding(kind):
    x = O.seeded((3000, 224), "normal", 5).cuda()[:, 16:208]  # row pitch 224
    out = torch.full((32, 128), 7.0, dtype=torch.float32, device="cuda")
    _run(x, kind, (5, 32, 2500, 96), out, out_pad=True)
    _check(out[0, :96], x[5:2505, 32:128], kind)
    assert bool((out[1:, :96] == 0).all()) and bool((out[:, 96:] == 7).all())


@pytest.mark.parametrize("h", [70, 4096])
def test_nan_and_infinity(h):
    x = O.seeded((h, 128), "normal", 7)
    x[h // 2, 3] = float("nan")
    x[1, 5] = float("inf")
    x[:, 9] = -float("inf")
    out = torch.zeros(1, 128, device="cuda")
    for kind in ("max", "sum"):
        _run(x.cuda(), kind, (0, 0, h, 128), out)
        got = out[0].cpu()
        assert bool(torch.isnan(got[3])) and float(got[5]) == float("inf")
        assert float(got[9]) == -float("inf")
        ok = torch.tensor([i for i in range(128) if i not in (3, 5, 9)])
        _check(got[ok], x[:, ok], kind)


def test_more_columns_than_one_launch_of_strips_holds():
    # 2^29 columns are 2^23 strips of 512 threads, one thread more than a launch
    # takes; one column strip fewer is the widest that the strips take
    for w in (2 ** 29 - 64, 2 ** 29):
        print(f"column strips 1x{w}", flush=True)
        x = torch.arange(w, dtype=torch.int32, device="cuda").remainder_(251).bfloat16().view(1, w)
        out = torch.zeros(1, w, device="cuda")
        _run(x, "max", (0, 0, 1, w), out)
        assert torch.equal(out, x.float())
        del x, out


def test_tall_and_narrow_operands_fill_the_chip():
    # the same 64 MB as 8192 x 4096 and as one strip: in eight shares of a strip
    # the tall one ran on 8 of 256 CUs, 15 times as long as the wide one
    def best(h, w):
        x = torch.ones(h, w, dtype=torch.bfloat16, device="cuda")
        out = torch.zeros(1, w, device="cuda")
        times = []
        for _ in range(8):
            start, end = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            torch.cuda._sleep(1000000)  # the host is ahead when the first launch starts
            start.record()
            for _ in range(4):
                _run(x, "sum", (0, 0, h, w), out)
            end.record()
            end.synchronize()
            times.append(start.elapsed_time(end))
        assert bool((out == h).all())
        return min(times)

    wide, tall = best(8192, 4096), best(2 ** 20, 32)
    print(f"column sums of 64 MB: wide {wide * 250:.1f} us, tall {tall * 250:.1f} us", flush=True)
    assert tall <= 5 * wide
