"""A failed wait is what Sampler reports, and it reads no output after it."""
from types import SimpleNamespace

import numpy as np
import pytest

import emel_hip as eh


@pytest.mark.parametrize("contiguous", [True, False])
def test_failed_wait_reads_no_outputs(contiguous):
    s = eh.Sampler.__new__(eh.Sampler)
    failed = eh.Status.INTERNAL
    s.stream = None
    s._lib = SimpleNamespace(emel_stream_synchronize=lambda stream: int(failed), emel_memcpy_dtoh=lambda *a: int(failed))
    s._local = SimpleNamespace(keep=None)
    host = np.zeros((2, 64), np.int32)
    s._local.keep = (host, host[0].ctypes.data, host[1].ctypes.data)
    # no reshape or cpu: an attempt to read raises
    out = SimpleNamespace(is_contiguous=lambda: contiguous, element_size=lambda: 4, numel=lambda: 8, data_ptr=lambda: 0)
    assert s._results(SimpleNamespace(selected_token_out=out, selected_score_out=out), 8) == (failed, None, None)
