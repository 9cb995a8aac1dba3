"""Extents past what one launch can index are accepted: HIP takes fewer than 2^32 work-items in a dimension, so a kernel
loops, or a call is launched in parts.  The operands here are larger than any memory; nothing runs."""
import pytest

import emel_hip as eh
from launch_recorder import Recorder, view

F16 = eh.DType.F16


@pytest.fixture(scope="module")
def rec():
    return Recorder()


def mul_mat(k, m, n, dtype=eh.DType.F32):
    rhs = [n, k, 1, 1] if dtype == eh.DType.F32 else [k, n, 1, 1]
    dst = [n, m, 1, 1] if dtype == eh.DType.F32 else [m, n, 1, 1]
    return eh.GenericEvent(eh.GenericRequest(eh.GenericOp.MUL_MAT, view(0, [k, m, 1, 1], dtype=dtype),
                                             view(1, rhs, dtype=dtype), None, view(2, dst, mut=True)))


def test_the_recorder_refuses_what_hip_refuses(rec):
    # 2^33 rows of one column, a lane each
    with pytest.raises(RuntimeError):
        rec.launches(eh.GenericEvent(eh.GenericRequest(eh.GenericOp.CUMSUM, view(0, [1, 1 << 33, 1, 1]), None, None,
                                                       view(1, [1, 1 << 33, 1, 1], mut=True))))


@pytest.mark.parametrize("k,m,n", [(64, 1 << 30, 1), (64, (1 << 30) + 5, 64), (64, 1, 1 << 31), (64, 16, 1 << 32), (256, 1 << 17, 1 << 18)])
@pytest.mark.parametrize("dtype", [eh.DType.F32, F16])
def test_mul_mat_extents(rec, k, m, n, dtype):
    got = rec.launches(mul_mat(k, m, n, dtype))
    if all("k_mm_any" in g.name or "k_mm_rows" in g.name for g in got):
        return  # these loop over their outputs
    tile = {"1, 1, 1, 1": 16, "1, 1, 2, 2": 32, "2, 2, 2, 2": 64}
    assert sum(g.grid * t * t for g in got for shape, t in tile.items() if f", {shape}, " in g.name) >= m * n


@pytest.mark.parametrize("event", [eh.OpAdd, eh.OpSub, eh.OpMul])
@pytest.mark.parametrize("n", [(1 << 34) - 1024, 1 << 34, (1 << 36) + 3])
def test_dense_binary_extents(rec, event, n):
    got, = rec.launches(event(view(0, [n, 1, 1, 1]), view(1, [n, 1, 1, 1]), view(2, [n, 1, 1, 1], mut=True)))
    per_lane = 32 if ", 8>" in got.name else 4
    assert got.grid * got.block * per_lane >= n // 4 * 4


@pytest.mark.parametrize("op,width,rows", [("RMS_NORM_BACK", 64, (1 << 29) + 1), ("RMS_NORM_BACK", 16, 1 << 30), ("SOFT_MAX_BACK", 32, 1 << 30),
                                           ("SOFT_MAX_BACK", 100, (1 << 32) - 64), ("SOFT_MAX_BACK", 128, (1 << 30) - 64)])
def test_back_rows_extents(rec, op, width, rows):
    params = eh.OpParams.i32(width) if op == "SOFT_MAX_BACK" else eh.OpParams.f32(1e-5)
    ne = [width, rows, 1, 1]
    got, = rec.launches(eh.GenericEvent(eh.GenericRequest(eh.GenericOp[op], view(0, ne), view(1, ne), None, view(2, ne, mut=True), params)))
    assert "k_back_rows" in got.name or got.grid * got.block >= rows  # a lane per row


@pytest.mark.parametrize("cols,rows", [(1027, 1 << 24), (1025, (1 << 26) - 4), (1023, (1 << 26) - 4)])
@pytest.mark.parametrize("event", ["soft_max", "soft_max_ext", "rms_norm", "rms_norm_mul"])
def test_ragged_rows_extents(rec, event, cols, rows):
    ne = [cols, rows, 1, 1]
    x, y = view(0, ne), view(1, ne, mut=True)
    got, = rec.launches({"soft_max": lambda: eh.OpSoftMax(x, y),
                         "soft_max_ext": lambda: eh.OpSoftMaxExt(x, None, 0.5, y),
                         "rms_norm": lambda: eh.OpRmsNorm(x, y, 1e-5),
                         "rms_norm_mul": lambda: eh.OpRmsNormMul(x, view(2, [cols, 1, 1, 1]), y, 1e-5)}[event]())
    assert got.grid * (4 if cols <= 1024 or "ragged" not in got.name else 1) >= rows


def test_products_of_2_to_the_27_outputs_take_two_launches(rec):
    for m, n in (((1 << 26) + 77, 1), (1, (1 << 27) + 77), (3, (1 << 27) + 5)):
        assert len(rec.launches(mul_mat(1, m, n))) == 2
