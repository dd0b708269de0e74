"""The fast product's split into bf16 planes (poorgrad_amd/csrc/gemm_mfma.hip)
where it can go wrong: the edges of every tile shape, k tails, odd extents of
outer-contiguous operands, unaligned bases, and the operands the planes cannot
carry (infinities, NaN, numbers that round to infinity, rows near the bottom
of the exponent range), which run on the f32 matrix cores instead.

Bound: each 16 k terms of an output are six matrix-core instructions of two
rounded additions each, a split along k adds at most 16 more, each rounding at
most 2^-24 of the running sum, itself at most sum |a b|; the three dropped
plane products and the remainders' own products stay below 2^-23 of it:
|error| <= (12 ceil(k / 16) + 18) 2^-24 sum |a b|."""
import numpy as np
import pytest
import torch

from tests.conftest import banner

pytestmark = pytest.mark.gpu


def product(hip, a, b):
    from poorgrad_amd import device

    out = device.gemm(a, b, hip.FAST)
    torch.cuda.synchronize()
    return out


def envelope(k):
    """The bound above, and never more than the contract's 1e-5."""
    return min((12 * -(-k // 16) + 18) * 2.0 ** -24, 1e-5)


def check(hip, a, b):
    """device.gemm over the views a, b against their f64 product; returns the
    relative 2-norm error."""
    got = product(hip, a, b).double()
    x, y = a.double(), b.double()
    want = x @ y
    bound = envelope(a.shape[1]) * (x.abs() @ y.abs())
    error = (got - want).abs()
    assert bool((error <= bound).all()), f"largest error over its bound {float((error / bound).nan_to_num().max())}"
    return float((got - want).norm() / want.norm())


def operand(seed, rows, columns, transposed, offset=0):
    """A [rows, columns] view whose unit-stride axis is the last (or, when
    `transposed`, the first), `offset` floats into its buffer."""
    g = torch.Generator().manual_seed(seed)
    flat = torch.randn(rows * columns + offset, generator=g).cuda()[offset:]
    return flat.view(columns, rows).t() if transposed else flat.view(rows, columns)


@pytest.mark.parametrize("m, k, n", [
    (1, 1, 1), (2, 3, 1), (1, 40, 65), (65, 15, 1), (63, 16, 65), (64, 17, 64), (65, 31, 63),   # 64-wide tiles
    (333, 64, 333), (1024, 70, 63), (62, 300, 1021), (127, 257, 129), (129, 33, 127),            # thin tiles, splits
    (1537, 1000, 777), (8192, 100, 769), (4095, 70, 2305),                                       # 128-wide tiles
    (4097, 50, 4095), (2047, 2049, 5631), (1025, 33, 50257)])                                    # 256-wide tiles
@pytest.mark.parametrize("left", [False, True])
@pytest.mark.parametrize("right", [False, True])
def test_split_product_edges(hip, m, k, n, left, right):
    banner(f"split product {m}x{k}x{n} {left} {right}")
    error = check(hip, operand(m + k, m, k, left, 1), operand(k + n, k, n, right, 3))
    # Random terms: the result's own rounding, at most 2^-24, and the chain's,
    # 1.55e-8 sqrt(k) (1.79e-8 sqrt(k) on the f32 matrix cores); without the
    # small plane products the error is 2^-17 or more.
    assert error <= 2.0 ** -24 + 1.8e-8 * k ** 0.5, error


@pytest.mark.parametrize("m, k, n", [(8193, 20, 8200), (8209, 20, 8179)])
def test_outputs_larger_than_the_last_level_cache(hip, m, k, n):
    """Just over 256 MB: 16-byte stores past the cache, and rows that allow none."""
    banner(f"streamed product {m}x{k}x{n}")
    assert 4 * m * n > 2 ** 28 and 4 * m * (n - 16) < 2 ** 28
    check(hip, operand(21, m, k, False), operand(22, k, n, True))


@pytest.mark.parametrize("m, k, n", [(70, 40, 66), (300, 200, 260)])
def test_split_product_of_unused_strides(hip, m, k, n):
    """Extent-1 axes leave their strides unused, whatever their value."""
    banner(f"unused strides {m}x{k}x{n}")
    column = operand(1, m, 5, False)[:, 2:3]          # [m, 1], rows 5 apart
    row = operand(2, 4, n, True)[1:2]                 # [1, n], columns 4 apart
    check(hip, column, row)
    check(hip, operand(3, 6, k, True)[4:5], operand(4, k, n, False))   # m = 1, k 6 apart
    check(hip, operand(5, m, k, False), operand(6, k, 7, False)[:, 3:4])  # n = 1, k 7 apart


def nonfinite_like(hip, a, b):
    """Where the f64 product of the same operands is infinite or NaN, so is
    the f32 one, with the same sign."""
    got = product(hip, a, b)
    want = a.double() @ b.double()
    assert bool((got.isnan() == want.isnan()).all())
    infinite = want.isinf()
    assert bool((got[infinite].double() == want[infinite]).all())
    return got, want


@pytest.mark.parametrize("m, k, n", [(96, 80, 112), (300, 1000, 260), (4096, 40, 4096)])
def test_nonfinite_operands(hip, m, k, n):
    banner(f"nonfinite operands {m}x{k}x{n}")
    a, b = operand(7, m, k, False).clone(), operand(8, k, n, False).clone()
    a[3, 5], a[m - 1, k - 1], b[7, n - 2] = float("inf"), float("nan"), -float("inf")
    b[5, :2] = 0.0
    a[:, 7] = a[:, 7].abs() + 0.5
    got, want = nonfinite_like(hip, a, b)
    finite = want.isfinite()
    bound = envelope(k) * (a.double().abs() @ b.double().abs())
    assert bool(((got.double() - want).abs()[finite] <= bound[finite]).all())
    nonfinite_like(hip, b.t(), a.t())


def test_numbers_that_round_to_infinity(hip):
    """The largest finite f32 rounds to an infinite bf16; its products are finite."""
    banner("numbers that round to infinity")
    largest = torch.finfo(torch.float32).max
    a = operand(9, 130, 48, False).clone()
    a[11] = 0.0
    a[11, 6], a[12, 40] = largest, -largest
    check(hip, a, operand(10, 48, 200, False) * 2.0 ** -4)


@pytest.mark.parametrize("small, large", [(2.0 ** -122, 2.0 ** 100), (2.0 ** -140, 2.0 ** 110)])
@pytest.mark.parametrize("m, k, n", [(100, 72, 90), (512, 512, 512), (2048, 64, 2048)])
def test_rows_near_the_bottom_of_the_exponent_range(hip, m, k, n, small, large):
    banner(f"small rows {m}x{k}x{n} {small}")
    a, b = operand(11, m, k, False).clone(), operand(12, k, n, True).clone() * large
    a[m // 2:m // 2 + 3] *= small
    a[0] = 0.0
    check(hip, a, b)
    check(hip, b.t(), a.t())


@pytest.mark.parametrize("exponent", [-109, -112, -118, -120, -126, -130, -135, -140, -148])
@pytest.mark.parametrize("m, k, n", [(64, 32, 64), (130, 70, 66), (96, 1000, 640), (2048, 64, 2048), (4096, 40, 4096)])
def test_rows_that_mix_magnitudes(hip, m, k, n, exponent):
    """Rows of one and of a number near the bottom of the exponent range, whose
    partners are zero and large: the planes drop the small number's low bits,
    and only its product reaches the output. Within the contract's 1e-5 sum
    |a b| in every orientation, as left and as right operand."""
    banner(f"mixed magnitudes {m}x{k}x{n} {exponent}")
    g = torch.Generator().manual_seed(m + k - exponent)
    small = (torch.rand(m, generator=g, dtype=torch.float64) + 1) * 2.0 ** exponent
    a, b = torch.zeros(m, k), torch.zeros(k, n)
    a[:, 0] = 1.0
    a[:, k - 3] = small.float()
    a[m // 2] = 0.0
    b[k - 3] = 2.0 ** min(-exponent, 120) * (torch.rand(n, generator=g) + 1)
    b[1, :] = torch.randn(n, generator=g)
    a, b = a.cuda(), b.cuda()
    x, y = a.double(), b.double()
    bound = 1e-5 * (x.abs() @ y.abs())
    for left in (a, a.t().contiguous().t()):
        for right in (b, b.t().contiguous().t()):
            for got in (product(hip, left, right), product(hip, right.t(), left.t()).t()):
                assert bool(((got.double() - x @ y).abs() <= bound).all())


@pytest.mark.parametrize("m, k, n, reach", [
    (2048, 2048, 2048, 1024), (1856, 4096, 6656, 512), (5312, 4032, 2496, 576), (640, 3392, 1408, 384),
    (1139, 3350, 748, 384), (3959, 7683, 344, 704), (58816, 1152, 576, 576)])
def test_ranges_are_as_short_as_the_f32_kernels(hip, m, k, n, reach):
    """Products that f32 matrix-core kernels sum in ranges of `reach` terms
    (their measured error over L random terms: 1.79e-8 sqrt(L) of the result,
    relative 2-norm) are no further from f64."""
    banner(f"ranges {m}x{k}x{n}")
    a, b = operand(31, m, k, False), operand(32, k, n, False)
    want = a.double() @ b.double()
    error = float((product(hip, a, b).double() - want).norm() / want.norm())
    assert error <= 1.79e-8 * reach ** 0.5, error


@pytest.mark.parametrize("exponent", [0, -118, -126])
@pytest.mark.parametrize("m, k, n", [(70, 1, 10), (2048, 1, 2048), (2048, 2, 2048), (300, 2, 70), (1030, 3, 1027),
                                     (8192, 3, 768)])
def test_products_of_few_terms(hip, m, k, n, exponent):
    """A chain of k fused multiply-adds rounds k times, each at most 2^-24 of
    sum |a b| (or half of 2^-149): one term is the correctly rounded product."""
    banner(f"few terms {m}x{k}x{n} {exponent}")
    a = operand(41, m, k, False) * 2.0 ** (exponent // 2)
    b = operand(42, k, n, True) * 2.0 ** (exponent - exponent // 2)
    x, y = a.double(), b.double()
    got = product(hip, a, b)
    if k == 1:
        assert bool((got == a * b).all())
    assert bool(((got.double() - x @ y).abs() <= k * (2.0 ** -24 * (x.abs() @ y.abs()) + 2.0 ** -150)).all())


@pytest.mark.parametrize("m, k, n", [(640, 1024, 1001), (96, 1024, 1023), (300, 2000, 70), (512, 512, 512)])
@pytest.mark.parametrize("extra, offset", [(0, 0), (4, 0), (3, 0), (4, 1)])
def test_ranges_into_spaced_rows(hip, m, k, n, extra, offset):
    """Products in several ranges of k, reduced into rows n + extra apart."""
    from poorgrad_amd import device

    banner(f"spaced rows {m}x{k}x{n} {extra} {offset}")
    a, b = operand(51, m, k, True), operand(52, k, n, False)
    held = torch.full((m * (n + extra) + offset,), 7.0, device="cuda")
    rows = held[offset:].view(m, n + extra)
    device.gemm(a, b, hip.FAST, out=rows[:, :n])
    torch.cuda.synchronize()
    x, y = a.double(), b.double()
    assert bool(((rows[:, :n].double() - x @ y).abs() <= 1e-5 * (x.abs() @ y.abs())).all())
    assert bool((rows[:, n:] == 7.0).all()) and bool((held[:offset] == 7.0).all())
    assert bool((rows[:, :n] == product(hip, a, b)).all())


@pytest.mark.parametrize("batch, heads, m, k, n", [(3, 5, 64, 333, 70), (2, 3, 100, 2000, 33), (2, 2, 65, 1025, 64)])
def test_ranges_of_two_level_batches(hip, batch, heads, m, k, n):
    """Attention's weights times values in several ranges of k: heads read
    through two batch strides and merged back into rows, whole quads or not."""
    from poorgrad_amd.topos import Tape
    from tests.program_util import run_device

    banner(f"two-level ranges {batch}x{heads} {m}x{k}x{n}")
    tape = Tape()
    weights = tape.input((batch * heads, m, k))
    values = tape.input((batch * k, heads * n)).reshape((batch, k, heads, n)).permute((0, 2, 1, 3))
    mixed = weights.matmul(values.reshape((batch * heads, k, n)))
    y = mixed.reshape((batch, heads, m, n)).permute((0, 2, 1, 3)).reshape((batch * m, heads * n))
    g = np.random.default_rng(m)
    w = g.standard_normal((batch * heads, m, k)).astype(np.float32)
    v = g.standard_normal((batch * k, heads * n)).astype(np.float32)
    got, program = run_device(tape, [y], [], {0: w, 1: v}, numerics=hip.FAST)
    lines = [line for line in program.describe.splitlines() if "gemm mfma" in line]
    assert len(lines) == 1 and " ranges" in lines[0] and program.info["launches"] == 1, program.describe
    wide = v.reshape(batch, k, heads, n).transpose(0, 2, 1, 3).reshape(batch * heads, k, n)

    def merged(x, z):
        t = np.matmul(x.astype(np.float64), z.astype(np.float64))
        return t.reshape(batch, heads, m, n).transpose(0, 2, 1, 3).reshape(batch * m, heads * n)

    assert (np.abs(got[y.id] - merged(w, wide)) <= 1e-5 * merged(np.abs(w), np.abs(wide))).all()


@pytest.mark.parametrize("left", [False, True])
@pytest.mark.parametrize("right", [False, True])
@pytest.mark.parametrize("m, k, n", [(2048, 16, 2048), (2048, 40, 2048), (4096, 64, 1024), (12544, 16, 72),
                                     (8192, 512, 4096), (512, 16, 512)])
def test_errors_do_not_add_up_over_rows_or_columns(hip, m, k, n, left, right):
    """Independent errors of the size the product has average out: the mean
    error of a row or a column lies within six standard deviations of zero."""
    banner(f"mean errors {m}x{k}x{n} {left} {right}")
    a, b = operand(61, m, k, left), operand(62, k, n, right)
    error = product(hip, a, b).double() - a.double() @ b.double()
    deviation = float(error.std())
    for axis, count in ((0, m), (1, n)):
        assert float(error.mean(axis).abs().max()) <= 6 * deviation / count ** 0.5
    assert abs(float(error.mean())) <= 6 * deviation / (m * n) ** 0.5


def test_zeros_are_positive(hip):
    """A product of zeros, signed or not, is +0."""
    banner("zeros")
    a = torch.zeros(70, 40, device="cuda")
    a[::2] = -0.0
    got = product(hip, a, -operand(13, 40, 70, False).abs())
    assert not bool(got.view(torch.int32).any())
    assert np.all(got.cpu().numpy() == 0.0)
