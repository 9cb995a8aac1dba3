"""What Sampler reports and what it leaves in flight when a copy of its results, or the wait for them, fails."""
from types import SimpleNamespace

import numpy as np
import pytest

import emel_hip as eh

FAILED = eh.Status.INTERNAL


class Library:
    """Copies and waits that fail where asked, in the order they were made."""

    def __init__(self, copies=(), wait=eh.Status.OK):
        self.copies, self.wait, self.calls = list(copies), wait, []

    def emel_memcpy_dtoh(self, dst, src, size, stream):
        self.calls.append("copy")
        return int(self.copies.pop(0))

    def emel_stream_synchronize(self, stream):
        self.calls.append("wait")
        return int(self.wait)


def results(lib, contiguous=True, rows=8):
    s = eh.Sampler.__new__(eh.Sampler)
    s.stream, s._lib = None, lib
    host = np.zeros((2, 64), np.int32)
    s._local = SimpleNamespace(keep=(host, host[0].ctypes.data, host[1].ctypes.data))
    # no reshape or cpu: an attempt to read raises
    out = SimpleNamespace(is_contiguous=lambda: contiguous, element_size=lambda: 4, numel=lambda: 8, data_ptr=lambda: 0)
    return s._results(SimpleNamespace(selected_token_out=out, selected_score_out=out), rows)


@pytest.mark.parametrize("contiguous", [True, False])
def test_failed_wait_reads_no_outputs(contiguous):
    lib = Library([eh.Status.OK, eh.Status.OK], FAILED)
    assert results(lib, contiguous) == (FAILED, None, None)
    assert lib.calls == ["copy", "copy", "wait"] if contiguous else ["wait"]


@pytest.mark.parametrize("copies", [[FAILED], [eh.Status.OK, FAILED]])
@pytest.mark.parametrize("wait", [eh.Status.OK, eh.Status.KERNEL_UNAVAILABLE])
def test_failed_copy_is_waited_for(copies, wait):
    # the copy before the failed one writes into a buffer that is handed on: it must be over, and the first error is reported
    lib = Library(copies, wait)
    assert results(lib) == (FAILED, None, None)
    assert lib.calls[-1] == "wait"
