"""Row programs over rows that are not whole quads (poorgrad_amd/csrc/codegen.cpp,
row_quads): four columns a point, the row's last, partial one from the row's last
four columns or lane by lane, bit for bit against the oracle, on both layouts (resident up to 2048 columns, streamed
beyond), at any base alignment, with special values in the partial quad, and
through programs whose inputs are broadcast along or across the row or
selected by index."""
import numpy as np
import pytest
import torch

import oracle
from poorgrad_amd import device
from tests.conftest import banner
from tests.gpu_util import assert_bitwise
from tests.program_util import run_device, run_oracle
from tests.test_rows_gpu import KINDS, expected_rows, kind_code

pytestmark = pytest.mark.gpu

# Below, at and above a quad; the widest resident row; one, two and three
# columns past a streamed slab; a lone row.
SHAPES = [(1, 9), (5, 10), (67, 11), (3, 33), (130, 333), (9, 2045), (2, 2047), (70, 2049), (33, 3470), (2, 5003),
          (1, 50257)]


def odd_rows(rows, columns, offset):
    g = oracle.Generator(rows * 7 + columns)
    x = g.normal(rows * columns, 3.0).reshape(rows, columns)
    if rows > 2:
        x[1, -1], x[2, -1] = np.inf, np.nan
        x[2, : columns // 2] = -0.0
    buffer = torch.full((rows * columns + offset,), float("nan"), device="cuda")
    view = buffer[offset:].view(rows, columns)
    view.copy_(torch.from_numpy(x))
    return x, view


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("rows, columns", SHAPES)
def test_odd_rows_bit_identical(hip, kind, rows, columns):
    banner(f"odd rows {kind} {rows}x{columns}")
    x, view = odd_rows(rows, columns, 1 + columns % 3)
    got = device.rows(kind_code(kind), view, hip.EXACT)
    torch.cuda.synchronize()
    assert_bitwise(got, expected_rows(kind_code(kind), x), f"{kind} {rows}x{columns}")


@pytest.mark.parametrize("rows, columns", SHAPES)
def test_odd_layer_norm_bit_identical(hip, rows, columns):
    banner(f"odd layer norm {rows}x{columns}")
    x, view = odd_rows(rows, columns, 3)
    g = oracle.Generator(columns)
    scale, shift = g.normal(columns, 1.0), g.normal(columns, 1.0)
    got = device.layer_norm(view, torch.from_numpy(scale).cuda(), torch.from_numpy(shift).cuda(), 1e-5, hip.EXACT)
    torch.cuda.synchronize()
    assert_bitwise(got, oracle.layer_norm_rows(x, scale, shift, 1e-5), f"layer norm {rows}x{columns}")


@pytest.mark.parametrize("columns", [9, 37, 2049])
def test_odd_row_programs_bit_identical(hip, columns):
    """A masked softmax (the mask broadcast over the leading axis) and a
    cross-entropy's row terms over a selection, through programs."""
    from poorgrad_amd.topos import Dense, Tape

    banner(f"odd row programs {columns}")
    g = oracle.Generator(columns)
    scores = g.normal(3 * 5 * columns, 2.0).reshape(3, 5, columns)
    mask = np.where(np.arange(columns)[None, :] <= np.arange(5)[:, None] + columns // 2, 0.0, -np.inf).astype(np.float32)
    labels = (np.arange(15) * 7 % columns).astype(np.int32)
    tape = Tape()
    s = tape.input((3, 5, columns))
    weights = (s + tape.leaf(Dense(mask)).broadcast_along(0, s)).softmax(2)
    flat = s.reshape((15, columns))
    targets = tape.selection_input(15, columns)
    terms = (targets * flat).sum_along(1) - flat.logsumexp(1)
    feeds = dict(dense={0: scores}, selections={1: (labels, 1.0)})
    want = run_oracle(tape, [weights, terms], [], **feeds)
    got, _ = run_device(tape, [weights, terms], [], numerics=hip.EXACT, **feeds)
    for root in (weights, terms):
        assert_bitwise(got[root.id], want[root.id], f"root {root.id}")


@pytest.mark.parametrize("rows, columns", [(40, 2049), (9000, 2305), (70000, 2051), (40, 4096)])
def test_many_folds_over_streamed_rows(hip, rows, columns):
    """Nine row sums in one pass, over slabs narrowed to fit LDS."""
    from poorgrad_amd.topos import Tape

    banner(f"many folds {rows}x{columns}")
    g = oracle.Generator(columns)
    x = g.normal(rows * columns, 1.0).reshape(rows, columns)
    scales = [g.normal(columns, 1.0) for _ in range(9)]
    tape = Tape()
    s = tape.input((rows, columns))
    total = None
    for _ in scales:
        part = (s * tape.parameter((columns,)).broadcast_along(0, s)).sum_along(1)
        total = part if total is None else total + part
    got, program = run_device(tape, [total], scales, dense={0: x}, numerics=hip.EXACT)
    assert " 9 folds, " in program.describe
    rows_checked = np.unique(np.r_[0:3, rows // 2, rows - 3:rows])
    want = None
    for scale in scales:
        terms = x[rows_checked] * scale
        part = terms[:, 0].copy()
        for j in range(1, columns):
            part = part + terms[:, j]
        want = part if want is None else want + part
    assert_bitwise(got[total.id][rows_checked], want, f"many folds {rows}x{columns}")


@pytest.mark.parametrize("rows, columns", [(1680, 50021), (330001, 257), (28001, 3001)])
def test_streamed_outputs_of_odd_rows(hip, rows, columns):
    """Outputs past the last-level cache's size, on both layouts, with a partial
    quad a row: sampled rows bit for bit, and nothing else written."""
    banner(f"streamed outputs {rows}x{columns}")
    assert 4 * rows * columns > 320 << 20
    g = torch.Generator("cuda").manual_seed(columns)
    x = torch.randn(rows, columns, generator=g, device="cuda")
    got = device.rows(hip.ROWS_SOFTMAX, x, hip.EXACT)
    picked = torch.tensor(sorted({0, 1, 2, 3, rows // 2, rows - 2, rows - 1}), device="cuda")
    assert_bitwise(got[picked], oracle.softmax_rows(x[picked].cpu().numpy()), f"softmax {rows}x{columns}")
    ones = got.double().sum(1)
    assert bool(((ones - 1).abs() < 1e-3).all())


@pytest.mark.parametrize("extent", [1, 3, 31, 32, 33, 383, 384, 385, 415, 416, 417, 767, 768, 769, 1151, 1155, 1537])
@pytest.mark.parametrize("outputs", [16, 20, 100])
def test_column_folds_at_their_tiles_edges(hip, extent, outputs):
    """Ordered column sums around tiles of 384 steps, folded 32 at a time."""
    from poorgrad_amd.topos import Tape

    banner(f"column fold {extent}x{outputs}")
    g = oracle.Generator(extent * 3 + outputs)
    x, y = (g.normal(extent * outputs, 1.0).reshape(extent, outputs) for _ in range(2))
    x[-1, 1], y[0, 2], x[0, 3] = np.inf, np.nan, -0.0
    tape = Tape()
    a, b = tape.input((extent, outputs)), tape.input((extent, outputs))
    sums = [a.sum_along(0), (a * b + a).sum_along(0)]
    feeds = {0: x, 1: y}
    want = run_oracle(tape, sums, [], dense=feeds)
    got, _ = run_device(tape, sums, [], dense=feeds, numerics=hip.EXACT)
    for s in sums:
        assert_bitwise(got[s.id], want[s.id], f"column fold {extent}x{outputs}")
