"""GPU parity of mul_mat's tiles (emel_generic_dispatch, MUL_MAT) with the oracle, bit for bit: the matrix
instructions' chains against the reference's sequential loop, at the edges of the tiles and of the staged blocks,
for every alignment the loads distinguish."""
import numpy as np
import pytest

import emel_hip as eh
import oracle as orc
from helpers import Pair, assert_bits_equal, rng

pytestmark = pytest.mark.gpu


def mul_mat(gpu, lhs, rhs, dst):
    want = orc.generic(eh.GenericOp.MUL_MAT, lhs.oview(), rhs.oview(), None, dst.oview(), b"", 0, 0, None)
    for p in (lhs, rhs, dst):
        p.to(gpu)
    req = eh.GenericRequest(eh.GenericOp.MUL_MAT, lhs.pview(), rhs.pview(), None, dst.pview(True))
    assert want == orc.OK and eh.Kernel().process_event(eh.GenericEvent(req)) == eh.Status.OK, eh.last_error()
    assert_bits_equal(dst.result(), dst.host, f"lhs {lhs.ne} rhs {rhs.ne}")


def values(seed, n, kind):
    g = rng(seed)
    x = g.standard_normal(n).astype(np.float32)
    if kind == "wide":  # exponents far apart: every order of additions gives other bits
        x = np.ldexp(x, g.integers(-12, 12, n)).astype(np.float32)
    elif kind == "special":
        at = g.integers(0, n, max(4, n // 2000))
        x[at] = np.array([np.inf, np.nan, -0.0, 1e-7], np.float32)[np.arange(at.size) % 4]
    return x


# k m n: one element, edges of the tiles (16 and 32 outputs, and one whole number of 64s) and of one or two of their
# blocks, k and n that are not whole vectors; longer inner dimensions in test_mul_mat_deep_tiles
SHAPES = [(1, 1, 1), (8, 16, 16), (520, 17, 16), (511, 15, 300), (96, 4096, 1), (1032, 40, 4), (264, 33, 65),
          (260, 33, 64), (128, 100, 31), (72, 2049, 1025), (67, 2050, 1023), (64, 2048, 1024)]


@pytest.mark.parametrize("kind", ["wide", "special"])
@pytest.mark.parametrize("k,m,n", SHAPES)
def test_mul_mat_f16_tiles(gpu, k, m, n, kind):
    lhs = values(k + m, k * m, kind).astype(np.float16).view(np.uint16)
    rhs = values(k + n, k * n, kind).astype(np.float16).view(np.uint16)
    mul_mat(gpu, Pair(lhs, [k, m, 1, 1]), Pair(rhs, [k, n, 1, 1]), Pair(np.zeros(m * n, np.float32), [m, n, 1, 1]))


@pytest.mark.parametrize("layout", ["dense", "lhs_columns", "rhs_columns", "padded"])
@pytest.mark.parametrize("k,m,n", SHAPES)
def test_mul_mat_f32_tiles(gpu, k, m, n, layout):
    kind = "special" if layout == "dense" else "wide"
    lhs, lnb, rhs, rnb = values(k + m, k * m, kind), None, values(k + n, k * n, kind), None
    if layout == "lhs_columns":  # lhs stored along m
        lnb = [4 * m, 4, 4 * k * m, 4 * k * m]
    elif layout == "rhs_columns":  # rhs stored along k
        rnb = [4 * k, 4, 4 * k * n, 4 * k * n]
    elif layout == "padded":  # rows of a longer stride, one float off a 16-byte boundary
        lhs, rhs = values(k + m, (k + 3) * m, kind), values(k + n, (n + 5) * k, kind)
        lnb, rnb = [4, 4 * (k + 3)] + [4 * (k + 3) * m] * 2, [4, 4 * (n + 5)] + [4 * (n + 5) * k] * 2
    mul_mat(gpu, Pair(lhs, [k, m, 1, 1], lnb), Pair(rhs, [n, k, 1, 1], rnb),
            Pair(np.zeros(m * n, np.float32), [n, m, 1, 1]))


# one dimension of 1 to 33 beside one long enough for whole rounds of 64x64 tiles
@pytest.mark.parametrize("k,m,n", [(264, 14850, 16), (257, 14850, 3), (72, 16390, 17), (300, 14849, 32), (64, 1, 14850),
                                   (260, 16391, 33), (48, 14850, 9)])
@pytest.mark.parametrize("dtype", ["f16", "f32"])
def test_mul_mat_narrow(gpu, k, m, n, dtype):
    lhs, rhs = values(k + m, k * m, "wide"), values(k + n, k * n, "wide")
    if dtype == "f16":
        lhs, rhs = (a.astype(np.float16).view(np.uint16) for a in (lhs, rhs))
        mul_mat(gpu, Pair(lhs, [k, m, 1, 1]), Pair(rhs, [k, n, 1, 1]), Pair(np.zeros(m * n, np.float32), [m, n, 1, 1]))
    else:
        mul_mat(gpu, Pair(lhs, [k, m, 1, 1]), Pair(rhs, [n, k, 1, 1]), Pair(np.zeros(m * n, np.float32), [n, m, 1, 1]))


# products that a lane per output takes, either side of a wave's columns, and transposed
@pytest.mark.parametrize("k,m,n", [(1, 1, 1), (1, 70, 63), (2, 300, 65), (4, 5000, 64), (7, 70001, 2), (16, 1, 70001), (32, 3, 40000)])
@pytest.mark.parametrize("layout", ["f16", "dense", "lhs_columns", "rhs_columns"])
def test_mul_mat_short_inner_dimension(gpu, k, m, n, layout):
    lhs, rhs, lnb, rnb = values(k + m, k * m, "special"), values(k + n, k * n, "wide"), None, None
    if layout == "f16":
        lhs, rhs = (a.astype(np.float16).view(np.uint16) for a in (lhs, rhs))
        mul_mat(gpu, Pair(lhs, [k, m, 1, 1]), Pair(rhs, [k, n, 1, 1]), Pair(np.zeros(m * n, np.float32), [m, n, 1, 1]))
        return
    if layout == "lhs_columns":
        lnb = [4 * m, 4, 4 * k * m, 4 * k * m]
    elif layout == "rhs_columns":
        rnb = [4 * k, 4, 4 * k * n, 4 * k * n]
    mul_mat(gpu, Pair(lhs, [k, m, 1, 1], lnb), Pair(rhs, [n, k, 1, 1], rnb), Pair(np.zeros(m * n, np.float32), [n, m, 1, 1]))


# Each tile's loop over blocks at work: the 64x64 tile's (blocks of 32, four in flight) from 161 inner elements, with
# every remainder of its four, whole vectors or not; 32x32 (blocks of 64, two) from 193; 16x16 (128, four) from 641.
# Rows and columns end inside a tile.
DEEP = [(64, 161, 1001, 963), (64, 200, 1001, 964), (64, 256, 1000, 964), (64, 260, 1001, 963), (64, 328, 1001, 964), (64, 385, 1001, 963),
        (32, 200, 1000, 300), (32, 301, 1000, 300), (32, 464, 999, 301), (16, 648, 33, 17), (16, 1501, 20, 5), (16, 1536, 50, 30)]


def deep_operands(k, m, n, layout):
    """(lhs [m, k], rhs [k, n]) as matrices, and the operands that hold them."""
    a, b = values(k + m, m * k, "wide").reshape(m, k), values(k + n, k * n, "wide").reshape(k, n)
    if layout == "f16":
        a, b = a.astype(np.float16), b.astype(np.float16)
        return a, b, Pair(a.reshape(-1).view(np.uint16), [k, m, 1, 1]), Pair(np.ascontiguousarray(b.T).reshape(-1).view(np.uint16), [k, n, 1, 1])
    lnb = rnb = None
    left, right = a, b
    if layout == "lhs_columns":
        left, lnb = np.ascontiguousarray(a.T), [4 * m, 4, 4 * k * m, 4 * k * m]
    elif layout == "rhs_columns":
        right, rnb = np.ascontiguousarray(b.T), [4 * k, 4, 4 * k * n, 4 * k * n]
    elif layout == "padded":
        left, lnb = np.pad(a, ((0, 0), (0, 3))), [4, 4 * (k + 3)] + [4 * (k + 3) * m] * 2
        right, rnb = np.pad(b, ((0, 0), (0, 5))), [4, 4 * (n + 5)] + [4 * (n + 5) * k] * 2
    return a, b, Pair(left.reshape(-1), [k, m, 1, 1], lnb), Pair(right.reshape(-1), [n, k, 1, 1], rnb)


@pytest.mark.parametrize("layout", ["f16", "dense", "lhs_columns", "rhs_columns", "padded"])
@pytest.mark.parametrize("tile,k,m,n", DEEP)
def test_mul_mat_deep_tiles(gpu, tile, k, m, n, layout):
    # The oracle's loop over all outputs takes ten seconds: it checks the bits of rows at the tiles' edges, every
    # column, and of columns at the edges, every row; 64 bits the rest.
    a, b, lhs, rhs = deep_operands(k, m, n, layout)
    f16 = layout == "f16"
    dst = Pair(np.full(m * n, 7.0, np.float32), [m, n, 1, 1] if f16 else [n, m, 1, 1]).to(gpu)
    req = eh.GenericRequest(eh.GenericOp.MUL_MAT, lhs.to(gpu).pview(), rhs.to(gpu).pview(), None, dst.pview(True))
    assert eh.Kernel().process_event(eh.GenericEvent(req)) == eh.Status.OK, eh.last_error()
    got = dst.result().reshape(n, m).T if f16 else dst.result().reshape(m, n)

    def oracle(rows, cols):
        x, z = a[rows], np.ascontiguousarray(b[:, cols])
        want = np.zeros(len(rows) * len(cols), np.float32)
        if f16:
            views = (orc.view(x.view(np.uint16).reshape(-1), [k, len(rows), 1, 1], None, orc.F16),
                     orc.view(np.ascontiguousarray(z.T).view(np.uint16).reshape(-1), [k, len(cols), 1, 1], None, orc.F16))
        else:
            views = orc.view(x.reshape(-1), [k, len(rows), 1, 1]), orc.view(z.reshape(-1), [len(cols), k, 1, 1])
        ne = [len(rows), len(cols), 1, 1] if f16 else [len(cols), len(rows), 1, 1]
        assert orc.generic(eh.GenericOp.MUL_MAT, *views, None, orc.view(want, ne), b"", 0, 0, None) == orc.OK
        return want.reshape(len(cols), len(rows)).T if f16 else want.reshape(len(rows), len(cols))

    edges = lambda d: sorted({i for i in (0, 1, 15, 16, 31, 32, 47, 63, 64, 65, d // 2, d - 2, d - 1) if i < d})  # noqa: E731
    rows, cols = edges(m), edges(n)
    what = f"{layout} {tile} k{k}"
    assert_bits_equal(got[rows], oracle(rows, list(range(n))), what + " rows")
    assert_bits_equal(np.ascontiguousarray(got[:, cols]), oracle(list(range(m)), cols), what + " columns")
    exact, size = a.astype(np.float64) @ b.astype(np.float64), np.abs(a).astype(np.float64) @ np.abs(b).astype(np.float64)
    # k roundings of the sum in 32 bits (F32), or in 64 with those of `exact` itself (F16), and the result's to 32
    bound = (2 * k * 2.0**-53 if f16 else k * 2.0**-24) * size + 2.0**-24 * np.abs(exact)
    assert (np.abs(got - exact) <= bound).all(), what


def test_mul_mat_f32_underflow_keeps_signed_zeros(gpu):
    # products that round to -0 and sums that end there: the staged blocks' padding must not turn them into +0
    k, m, n = 5, 20, 18
    lhs = np.full(k * m, -1e-30, np.float32)
    lhs[: k * 3] = 1e-30
    rhs = np.full(n * k, 1e-30, np.float32)
    mul_mat(gpu, Pair(lhs, [k, m, 1, 1]), Pair(rhs, [n, k, 1, 1]), Pair(np.ones(m * n, np.float32), [n, m, 1, 1]))


def test_mul_mat_f32_rows_far_apart(gpu):
    # rows 32 MiB apart: past the tiles' 32-bit offsets
    k, m, n, row = 6, 3, 4, (1 << 23) + 4
    lhs = np.zeros(row * m, np.float32)
    lhs.reshape(m, row)[:, :k] = values(1, k * m, "wide").reshape(m, k)
    mul_mat(gpu, Pair(lhs, [k, m, 1, 1], [4, 4 * row, 4 * row * m, 4 * row * m]),
            Pair(values(2, k * n, "wide"), [n, k, 1, 1]), Pair(np.zeros(m * n, np.float32), [n, m, 1, 1]))


@pytest.mark.parametrize("m,n", [((1 << 26) + 77, 1), (1, (1 << 27) + 77), (3, (1 << 27) + 5)])
def test_mul_mat_more_outputs_than_one_launch(gpu, m, n):
    # k = 1: every output is one product, rounded, plus +0
    import torch

    g = torch.Generator(device=gpu).manual_seed(m)
    a, b = torch.randn(m, device=gpu, generator=g), torch.randn(n, device=gpu, generator=g)
    y = torch.full((m * n,), 7.0, device=gpu)
    dense = lambda t, ne, cls=eh.TensorView: cls(t, eh.Layout.dense(eh.DType.F32, ne))  # noqa: E731
    req = eh.GenericRequest(eh.GenericOp.MUL_MAT, dense(a, [1, m, 1, 1]), dense(b, [n, 1, 1, 1]), None,
                            dense(y, [n, m, 1, 1], eh.TensorViewMut))
    assert eh.Kernel().process_event(eh.GenericEvent(req)) == eh.Status.OK, eh.last_error()
    assert torch.equal(y.view(m, n), a[:, None] * b[None, :])


def argmax(gpu, lhs, rhs):
    dst, idx = Pair(np.zeros(1, np.float32), [1, 1, 1, 1]).to(gpu), np.full(1, -7, np.int32)
    want = orc.generic(eh.GenericOp.MUL_MAT_ARGMAX, lhs.oview(), rhs.oview(), None, dst.oview(), b"", 0, 0, idx)
    index = Pair(np.full(1, -7, np.int32), [1, 1, 1, 1]).to(gpu)
    req = eh.GenericRequest(eh.GenericOp.MUL_MAT_ARGMAX, lhs.to(gpu).pview(), rhs.to(gpu).pview(), None,
                            dst.pview(True)).with_index_out(index.dev)
    assert want == orc.OK and eh.Kernel().process_event(eh.GenericEvent(req)) == eh.Status.OK, eh.last_error()
    assert_bits_equal(dst.result(), dst.host, "value")
    assert int(index.dev.cpu()[0]) == int(idx[0])


# k m: row tails and tile tails of each row count per wave (16, 32, 64 rows; tiles of 128, 64, 32 columns), more row
# blocks than workgroups, and rows that are not whole vectors
@pytest.mark.parametrize("k,m", [(4, 1), (132, 15), (260, 33), (512, 17), (68, 65600), (36, 131137), (8, 600001), (37, 50),
                                 (4, 70000), (8, 11999), (12, 12001), (8, 131072)])
@pytest.mark.parametrize("case", ["plain", "tie", "zeros", "nan", "nan_first", "all_nan"])
def test_mul_mat_argmax_rows(gpu, k, m, case):
    w, h = values(k * m, k * m, "wide"), values(k, k, "wide")
    rows = w.reshape(m, k)
    if case == "tie":  # the greatest row, again later
        rows[m // 2] = np.abs(w).max() * np.sign(h)
        rows[m - 1] = rows[m // 2]
    elif case == "zeros":  # every dot +0 or -0: the first row wins with its own sign
        rows[:] = np.where(np.arange(m) % 2 == 0, np.float32(-1e-30), np.float32(1e-30))[:, None]
        h[:] = np.float32(1e-30)
    elif case == "nan":
        rows[m - 1, k // 2] = np.nan
    elif case == "nan_first":
        rows[0, 0] = np.nan
    elif case == "all_nan":
        h[0] = np.nan
    argmax(gpu, Pair(w, [k, m, 1, 1]), Pair(h, [k, 1, 1, 1]))


@pytest.mark.parametrize("k,m", [(4, 1), (260, 33), (132, 4097), (36, 131137), (4, 16390), (8, 16385)])
def test_mul_mat_f32_one_column(gpu, k, m):
    # rhs and dst columns apart, lhs rows padded
    lhs, rhs = values(k + m, (k + 8) * m, "special"), values(k, k, "wide")
    mul_mat(gpu, Pair(lhs, [k, m, 1, 1], [4, 4 * (k + 8)] + [4 * (k + 8) * m] * 2), Pair(rhs, [1, k, 1, 1]),
            Pair(np.zeros(3 * m, np.float32), [1, m, 1, 1], [4, 12, 12 * m, 12 * m]))
