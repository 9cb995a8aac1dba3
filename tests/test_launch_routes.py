"""Which kernel a call takes, where the choice was measured: nothing runs, the launches are recorded."""
import re

import pytest

import emel_hip as eh
from launch_recorder import Recorder, view

F32, F16 = eh.DType.F32, eh.DType.F16


@pytest.fixture(scope="module")
def rec():
    return Recorder()


def mul_mat(rec, k, m, n, dtype=F32, layout="dense"):
    """The kernel of one product: the tile's edge, "lane" (k_mm_any) or "rows"."""
    lnb = rnb = None
    if layout == "lhs_columns":
        lnb = [4 * m, 4, 4 * k * m, 4 * k * m]
    elif layout == "rhs_columns":
        rnb = [4 * k, 4, 4 * k * n, 4 * k * n]
    rhs, dst = ([n, k, 1, 1], [n, m, 1, 1]) if dtype == F32 else ([k, n, 1, 1], [m, n, 1, 1])
    got, = rec.launches(eh.GenericEvent(eh.GenericRequest(eh.GenericOp.MUL_MAT, view(0, [k, m, 1, 1], lnb, dtype),
                                                          view(1, rhs, rnb, dtype), None, view(2, dst, mut=True))))
    tile = re.search(r"k_mm_tile<\w+, \w+, \w+, \w+, (\d), (\d), (\d), (\d),", got.name)
    if tile:
        fi, fj, wi, wj = map(int, tile.groups())
        assert fi * wi == fj * wj
        return 16 * fi * wi
    return "lane" if "k_mm_any" in got.name else "rows"


@pytest.mark.parametrize("m", [14800, 16384, 32000, 65536, 128256, 151936])
@pytest.mark.parametrize("n", [1, 4, 16])
def test_mul_mat_narrow_f16_takes_small_tiles(rec, m, n):
    assert mul_mat(rec, 4096, m, n, F16) == 16
    assert mul_mat(rec, 4096, n, m, F16) == 16  # the narrow side first
    assert mul_mat(rec, 4095, m, n, F16) == 32  # halves gathered one by one
    assert mul_mat(rec, 64, m, n, F16) == 32 and mul_mat(rec, 48, m, n, F16) == 64


@pytest.mark.parametrize("m", [16384, 32000, 151936])
@pytest.mark.parametrize("n", [2, 16, 17, 32])
def test_mul_mat_narrow_takes_32_wide_tiles(rec, m, n):
    assert mul_mat(rec, 4096, m, n) == mul_mat(rec, 4096, n, m) == 32
    if n > 16:
        assert mul_mat(rec, 4096, m, n, F16) == 32
    # a transposed operand is gathered: the larger tile reads whole lines of it
    assert mul_mat(rec, 4096, m, n, layout="lhs_columns") == 64
    assert mul_mat(rec, 4096, m, n, layout="rhs_columns") == 64


def test_mul_mat_wide_products_keep_their_tiles(rec):
    assert mul_mat(rec, 4096, 4096, 512, F16) == mul_mat(rec, 4096, 16384, 48) == mul_mat(rec, 4096, 4096, 256) == 64
    assert mul_mat(rec, 704, 10533, 283, F16) == mul_mat(rec, 4096, 4096, 64) == 32
    assert mul_mat(rec, 4096, 4096, 16) == mul_mat(rec, 4096, 4096, 1, F16) == 16
    assert mul_mat(rec, 4096, 32000, 1) == "rows"


@pytest.mark.parametrize("dtype", [F32, F16])
def test_mul_mat_short_inner_dimension_takes_lanes(rec, dtype):
    for k, m, n in [(1, 1, 1), (1, 1 << 20, 4), (1, 4, 1 << 20), (1, 1 << 24, 1), (1, 4096, 4096), (2, 1 << 20, 2), (4, 1 << 20, 3),
                    (7, 300000, 2), (16, 1, 1 << 20)]:
        assert mul_mat(rec, k, m, n, dtype) == "lane", (k, m, n)
    for k, m, n in [(8, 4096, 4096), (16, 4096, 512), (32, 512, 512), (64, 64, 64), (33, 1 << 20, 2)]:
        assert mul_mat(rec, k, m, n, dtype) != "lane", (k, m, n)


def test_mul_mat_short_inner_dimension_of_transposed_operands(rec):
    # neighbouring lanes read neighbouring elements
    assert mul_mat(rec, 32, 1 << 20, 1, layout="lhs_columns") == mul_mat(rec, 512, 1 << 20, 1, layout="lhs_columns") == "lane"
    assert mul_mat(rec, 64, 1, 1 << 20) == "lane" and mul_mat(rec, 256, 1, 1 << 20) == 32
    assert mul_mat(rec, 256, 151936, 1, layout="lhs_columns") == 64
    assert mul_mat(rec, 8, 1, 1 << 22, layout="rhs_columns") == "lane"
    assert mul_mat(rec, 32, 2, 1 << 20, layout="rhs_columns") == 64  # 128 bytes apart


def argmax(rec, k, m):
    req = eh.GenericRequest(eh.GenericOp.MUL_MAT_ARGMAX, view(0, [k, m, 1, 1]), view(1, [k, 1, 1, 1]), None,
                            view(2, [1, 1, 1, 1], mut=True))

    class Index:  # what with_index_out asks of a tensor
        def data_ptr(self):
            return 3 << 43

        def element_size(self):
            return 4

    req.with_index_out(Index())
    first, last = rec.launches(eh.GenericEvent(req))
    assert "k_mm_argmax_final" in last.name
    return "rows" if "k_mm_rows" in first.name else "walk"


def test_rows_of_four_are_walked(rec):
    for m in (1, 1000, 16384, 1 << 20, 1 << 24):
        assert argmax(rec, 4, m) == "walk" and mul_mat(rec, 4, m, 1) == "lane"
    assert mul_mat(rec, 8, 16384, 1) == mul_mat(rec, 16, 1 << 20, 1) == "rows"
    for k in (8, 12):
        assert [argmax(rec, k, m) for m in (1000, 11999, 12000, 65536, 1 << 17, 1 << 20)] == ["rows", "rows", "walk", "walk", "rows", "rows"]
    assert argmax(rec, 16, 24000) == argmax(rec, 4096, 151936) == "rows"


def back(rec, op, width, rows, offset=0):
    ne = [width, rows, 1, 1]
    params = eh.OpParams.i32(width) if op == "SOFT_MAX_BACK" else eh.OpParams.f32(1e-5)
    got, = rec.launches(eh.GenericEvent(eh.GenericRequest(eh.GenericOp[op], view(0, ne, offset=offset), view(1, ne), None,
                                                          view(2, ne, mut=True), params)))
    return "groups" if "k_back_rows" in got.name else "lanes"


@pytest.mark.parametrize("op,lanes,groups", [
    ("SOFT_MAX_BACK", [(1, 1), (1, 10000000), (3, 1000), (7, 1), (7, 1000000), (4, 60000), (9, 512), (10, 1000000), (13, 100000)],
     [(4, 30000), (8, 100), (8, 1000000), (9, 300), (13, 300), (13, 300000), (11, 1000000), (14, 1), (15, 30000), (17, 1000), (512, 16384)]),
    ("RMS_NORM_BACK", [(1, 1), (2, 10000000), (4, 1), (7, 100), (9, 300), (15, 1000000), (8, 30000), (12, 100000), (17, 60000), (23, 100000)],
     [(8, 1000), (12, 10000), (9, 100), (15, 100), (16, 1), (16, 100000), (17, 10000), (17, 300000), (24, 60000), (4096, 512)])])
def test_narrow_gradient_rows_take_lanes(rec, op, lanes, groups):
    assert [(w, r) for w, r in lanes if back(rec, op, w, r) != "lanes"] == []
    assert [(w, r) for w, r in groups if back(rec, op, w, r) != "groups"] == []


def test_narrow_gradient_rows_off_16_bytes(rec):
    # loaded one by one, as odd widths
    assert back(rec, "SOFT_MAX_BACK", 8, 1000, offset=4) == back(rec, "RMS_NORM_BACK", 16, 60000, offset=4) == "lanes"
    assert back(rec, "SOFT_MAX_BACK", 16, 1000, offset=4) == back(rec, "RMS_NORM_BACK", 24, 60000, offset=4) == "groups"


@pytest.mark.parametrize("width,rows", [(17, 4097), (18, 30001), (1023, 2500), (513, 3100)])
def test_gradient_rows_of_odd_widths_run_in_one_round(rec, width, rows):
    ne = [width, rows, 1, 1]
    got, = rec.launches(eh.GenericEvent(eh.GenericRequest(eh.GenericOp.SOFT_MAX_BACK, view(0, ne), view(1, ne), None,
                                                          view(2, ne, mut=True), eh.OpParams.i32(width))))
    assert "k_back_rows" in got.name and got.grid <= 512  # two workgroups on each of 256 CUs


def eights(rec, op, mb):
    """Whether the dense copy or binary that moves `mb` MB takes eight float4 per lane."""
    n = int(mb * 1e6 / (8 if op == "copy" else 12)) // 4 * 4
    a, b, y = view(0, [n, 1, 1, 1]), view(1, [n, 1, 1, 1]), view(2, [n, 1, 1, 1], mut=True)
    got, = rec.launches({"copy": lambda: eh.DenseOpDup(a.ptr, y.ptr, n, n), "add": lambda: eh.OpAdd(a, b, y), "sub": lambda: eh.OpSub(a, b, y),
                         "mul": lambda: eh.OpMul(a, b, y)}[op]())
    return ", 8>" in got.name


@pytest.mark.parametrize("op,few,many", [
    ("copy", [1, 16, 20, 26, 34, 36, 51, 120, 150], [28.5, 33, 40, 50, 60, 67, 70, 80, 95, 110, 117]),
    ("add", [1, 12, 25, 26, 40, 51, 60, 76, 83, 90, 95, 101, 104, 115, 125, 200], [46, 50, 67.6, 70, 75, 100]),
    ("sub", [55, 80, 101], [46, 50, 75]), ("mul", [55, 80, 101], [46, 50, 75])])
def test_dense_streams_take_eights_where_their_last_round_is_full(rec, op, few, many):
    assert [mb for mb in few if eights(rec, op, mb)] == []
    assert [mb for mb in many if not eights(rec, op, mb)] == []


def test_the_deep_products_reach_their_tiles(rec):
    from test_gpu_mulmat import DEEP

    blocks = {16: (128, 4), 32: (64, 2), 64: (32, 4)}  # elements per block, blocks in flight
    for tile, k, m, n in DEEP:
        size, flight = blocks[tile]
        assert -(-k // size) > flight + 1, (tile, k)  # the loop over blocks runs
        for dtype in (F32, F16):
            assert mul_mat(rec, k, m, n, dtype) == tile, (tile, k, m, n)
        for layout in ("lhs_columns", "rhs_columns"):
            assert mul_mat(rec, k, m, n, layout=layout) == tile
    assert {-(-k // 32) % 4 for tile, k, _, _ in DEEP if tile == 64} == {0, 1, 2, 3}
