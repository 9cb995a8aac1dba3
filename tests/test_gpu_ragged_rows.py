"""GPU parity of soft_max, soft_max_ext and rms_norm (+weight) rows of any width and alignment with the oracle: partial
last vectors at every width class of the row kernels, rows and masks that start off their vectors' boundaries, rows with
non-finite values, and the bytes around the destination left alone.  1e-5 relative, as for whole vectors: the f64 sums
run as a tree."""
import numpy as np
import pytest

import emel_hip as eh
import oracle as orc
from helpers import assert_close_rel, normal, rng

pytestmark = pytest.mark.gpu
RTOL = 1e-5
WIDTHS = [4, 5, 7, 255, 257, 511, 514, 1023, 1025, 2047, 2050, 4093, 4099, 8191, 16383, 16385, 20001]


class Off:
    """A device buffer whose data starts `off` elements past a 16-byte boundary, with guards on both sides."""

    def __init__(self, gpu, host, off):
        import torch

        self.n, self.off = host.size, off
        self.t = torch.from_numpy(np.concatenate([np.full(4 + off, 77, host.dtype), host, np.full(9, 77, host.dtype)])).to(gpu)

    def view(self, ne, dtype=0, mut=False):
        cls = eh.TensorViewMut if mut else eh.TensorView
        return cls(self.t[4 + self.off: 4 + self.off + self.n], eh.Layout.dense(dtype, ne), self.n * self.t.element_size())

    def result(self):
        a = self.t.cpu().numpy()
        assert (a[: 4 + self.off] == 77).all() and (a[4 + self.off + self.n:] == 77).all(), "wrote outside dst"
        return a[4 + self.off: 4 + self.off + self.n]


def close(got, want, what):
    assert (np.isnan(got) == np.isnan(want)).all(), what
    assert_close_rel(got, want, RTOL, what)


@pytest.mark.parametrize("off", [0, 1, 2])
@pytest.mark.parametrize("cols", WIDTHS)
def test_ragged_soft_max_ext(gpu, cols, off):
    ne = [cols, 3, 2, 2]
    n = int(np.prod(ne))
    x = normal(cols, n, 2.0)
    x[cols * 4] = np.nan
    x[cols * 5 - 1] = np.inf  # a row's last column
    x[cols * 7 - 1] = 100.0   # ... holds the maximum
    mask = (rng(cols).standard_normal(cols * 3 * 2) * 2).astype(np.float16)
    mask[rng(cols + 1).random(mask.size) < 0.3] = np.float16(-np.inf)
    mask.reshape(-1, cols)[:, 0] = 0
    mask.reshape(-1, cols)[1, :] = np.float16(-np.inf)  # a row with nothing left
    want = np.zeros_like(x)
    assert orc.soft_max_ext(orc.view(x, ne), orc.view(mask.view(np.uint16), [cols, 3, 2, 1], None, orc.F16), 0.5,
                            orc.view(want, ne)) == orc.OK
    xo, yo, mo = Off(gpu, x, off), Off(gpu, np.zeros_like(x), (off + 1) % 4), Off(gpu, mask.view(np.int16), off)
    assert eh.Kernel().process_event(eh.OpSoftMaxExt(xo.view(ne), mo.view([cols, 3, 2, 1], eh.DType.F16), 0.5,
                                                     yo.view(ne, mut=True))) == eh.Status.OK, eh.last_error()
    close(yo.result(), want, f"soft_max_ext {cols}")


@pytest.mark.parametrize("cols", WIDTHS)
def test_ragged_soft_max_and_rms_norm(gpu, cols):
    ne = [cols, 5, 1, 1]
    x = normal(cols + 1, 5 * cols, 3.0)
    x[cols * 2 - 1] = -np.inf
    w = normal(cols + 2, cols)
    k = eh.Kernel()
    for name in ("soft_max", "rms_norm", "rms_norm_mul"):
        want = np.zeros_like(x)
        xo, wo, yo = Off(gpu, x, 1), Off(gpu, w, 3), Off(gpu, np.zeros_like(x), 2)
        if name == "soft_max":
            ev, st = eh.OpSoftMax(xo.view(ne), yo.view(ne, mut=True)), orc.soft_max(orc.view(x, ne), orc.view(want, ne))
        elif name == "rms_norm":
            ev, st = eh.OpRmsNorm(xo.view(ne), yo.view(ne, mut=True), 1e-5), orc.rms_norm(orc.view(x, ne), orc.view(want, ne), 1e-5)
        else:
            ev = eh.OpRmsNormMul(xo.view(ne), wo.view([cols, 1, 1, 1]), yo.view(ne, mut=True), 1e-5)
            st = orc.rms_norm_mul(orc.view(x, ne), orc.view(w, [cols, 1, 1, 1]), orc.view(want, ne), 1e-5)
        assert st == orc.OK and k.process_event(ev) == eh.Status.OK, eh.last_error()
        close(yo.result(), want, f"{name} {cols}")


def test_ragged_rows_in_place(gpu):
    cols, ne = 1027, [1027, 9, 1, 1]
    x = normal(3, 9 * cols)
    want = np.zeros_like(x)
    assert orc.soft_max(orc.view(x, ne), orc.view(want, ne)) == orc.OK
    b = Off(gpu, x, 1)
    assert eh.Kernel().process_event(eh.OpSoftMax(b.view(ne), b.view(ne, mut=True))) == eh.Status.OK, eh.last_error()
    close(b.result(), want, "in place")
