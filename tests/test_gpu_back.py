"""GPU parity of soft_max_back and rms_norm_back over dense operands with the oracle, bit for bit: widths around the
chains' steps, the tile of 8192 elements and its groups of rows, unaligned buffers, and results written over an input."""
import numpy as np
import pytest

import emel_hip as eh
import oracle as orc
from helpers import assert_bits_equal, normal, rng
from test_gpu_generic import f32p, i32p

pytestmark = pytest.mark.gpu
G = eh.GenericOp


def run(gpu, op, x, g, ne, params, into=None, offset=0):
    import torch

    want = np.zeros_like(x)
    assert orc.generic(op, orc.view(x, ne), orc.view(g, ne), None, orc.view(want, ne), params, len(params), 0, None) == orc.OK
    lay = eh.Layout.dense(0, ne)

    def dev(a):  # `offset` floats past a 16-byte boundary
        t = torch.zeros(a.size + offset, device=gpu)
        t[offset:] = torch.from_numpy(a).to(gpu)
        return t[offset:]

    xd, gd = dev(x), dev(g)
    yd = {None: dev(np.full_like(x, 7.0)), "x": xd, "g": gd}[into]
    req = eh.GenericRequest(op, eh.TensorView(xd, lay), eh.TensorView(gd, lay), None, eh.TensorViewMut(yd, lay),
                            eh.OpParams(params))
    assert eh.Kernel().process_event(eh.GenericEvent(req)) == eh.Status.OK, eh.last_error()
    assert_bits_equal(yd.cpu().numpy(), want, f"{G(op).name} {ne}")


# width, rows: partial chain steps, rows that are not whole vectors, groups of rows with a short last one, one row per
# workgroup, exactly a tile, rows of several tiles
SHAPES = [(1, 3), (3, 70), (5, 40000), (33, 1031), (64, 600), (127, 5), (128, 70000), (512, 1030), (700, 513), (2047, 9),
          (2050, 3000), (4096, 7), (8192, 3), (8193, 3), (20000, 2)]


@pytest.mark.parametrize("op", [G.SOFT_MAX_BACK, G.RMS_NORM_BACK])
@pytest.mark.parametrize("width,rows", SHAPES)
@pytest.mark.parametrize("offset", [0, 1])
def test_back_rows(gpu, op, width, rows, offset):
    n = width * rows
    x, g = normal(width, n), normal(rows, n)
    if offset:  # every order of additions gives other bits; zeros of both signs and non-finite rows
        x = np.ldexp(x, rng(3).integers(-12, 12, n)).astype(np.float32)
        x[rng(4).integers(0, n, 3)] = [np.inf, np.nan, -0.0]
        g[rng(5).integers(0, n, 2)] = [-0.0, 0.0]
    params = i32p(width) if op == G.SOFT_MAX_BACK else f32p(1e-5)
    run(gpu, op, x, g, [width, rows, 1, 1], params, offset=offset)


# either side of what takes a lane per row
@pytest.mark.parametrize("op", [G.SOFT_MAX_BACK, G.RMS_NORM_BACK])
@pytest.mark.parametrize("width,rows", [(4, 32767), (4, 32768), (7, 1000), (8, 16383), (8, 16384), (9, 255), (9, 512), (12, 16385),
                                        (11, 190650), (11, 190651), (13, 511), (13, 512), (14, 600), (15, 65537), (16, 20000),
                                        (17, 4097), (17, 16384), (18, 30001), (23, 131072)])
@pytest.mark.parametrize("offset", [0, 1])
def test_narrow_back_rows(gpu, op, width, rows, offset):
    n = width * rows
    x = np.ldexp(normal(width, n), rng(9).integers(-12, 12, n)).astype(np.float32)
    run(gpu, op, x, normal(rows, n), [width, rows, 1, 1], i32p(width) if op == G.SOFT_MAX_BACK else f32p(1e-5), offset=offset)


@pytest.mark.parametrize("op", [G.SOFT_MAX_BACK, G.RMS_NORM_BACK])
@pytest.mark.parametrize("into", ["x", "g"])
@pytest.mark.parametrize("width", [96, 8448])
def test_back_rows_in_place(gpu, op, into, width):
    x, g = normal(1, width * 6), normal(2, width * 6)
    run(gpu, op, x, g, [width, 3, 2, 1], i32p(width) if op == G.SOFT_MAX_BACK else f32p(0.0), into=into)


@pytest.mark.parametrize("row", [6, 21, 60, 420])
def test_soft_max_back_rows_of_ordinals(gpu, row):
    # rows are runs of ordinals, whatever the extents
    x, g = normal(6, 840), normal(7, 840)
    run(gpu, G.SOFT_MAX_BACK, x, g, [6, 10, 7, 2], i32p(row))


# either side of what is staged as doubles: width 512, a CU's LDS for two workgroups and for one, 512 workgroups,
# groups of rows
@pytest.mark.parametrize("width,rows", [(508, 40), (512, 40), (4928, 257), (4932, 257), (4932, 256), (4096, 512), (2050, 1025),
                                        (1024, 2000), (1023, 2000)])
def test_rms_norm_back_staging(gpu, width, rows):
    n = width * rows
    x = np.ldexp(normal(width, n), rng(8).integers(-12, 12, n)).astype(np.float32)
    run(gpu, G.RMS_NORM_BACK, x, normal(rows, n), [width, rows, 1, 1], f32p(1e-5))
