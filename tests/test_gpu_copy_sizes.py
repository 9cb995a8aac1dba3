"""The dense copy and binary streams at sizes around those where they change their shape (rounds of 256 workgroups of 8192
elements: the copy from 400 of 512 to 1792 workgroups, the sum from 446 to 768), with tails."""
import pytest
import torch

import emel_hip as eh

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 3, 1023, 3499999, 3500000, 3500002, 3502081, 3750000, 3750001, 8750000, 8750003, 14500000, 14500001, 14502051,
                               3268608, 3268612, 3653628, 3645440, 3645444, 4194304, 4194308, 6291456, 6291459, 6291460, 14680064, 14680068])
def test_copy_and_add_sizes(gpu, n):
    k = eh.Kernel()
    x = torch.arange(n, device=gpu, dtype=torch.int32).add_(0x3f000001).view(torch.float32)
    y = torch.full((n + 8,), -1.0, device=gpu)
    assert k.process_event(eh.DenseOpDup(x, y, output_len=n)) == eh.Status.OK, eh.last_error()
    assert torch.equal(y[:n].view(torch.int32), x.view(torch.int32)) and bool((y[n:] == -1.0).all())
    assert k.process_event(eh.DenseOpAdd(x, x, y, output_len=n)) == eh.Status.OK, eh.last_error()
    assert torch.equal(y[:n], x + x) and bool((y[n:] == -1.0).all())
