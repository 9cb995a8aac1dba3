"""The selections that Sampler hands back: they are what the call left in selected_token_out and selected_score_out, row
by row, for more rows than one result buffer held before, for tensors that are views, and from several threads."""
import threading

import numpy as np
import pytest
import torch

import emel_hip as eh

pytestmark = pytest.mark.gpu


def sample(gpu, sampler, rows, seed, token=None, score=None, card=600, k=5):
    g = np.random.Generator(np.random.PCG64(seed))
    x = g.standard_normal((rows, card)).astype(np.float32)
    if rows > 2:
        x[2] = np.nan  # no valid result
    i32 = dict(dtype=torch.int32, device=gpu)
    token = torch.full((rows,), -3, **i32) if token is None else token
    score = torch.zeros(rows, device=gpu) if score is None else score
    req = eh.SampleTemperatureTopK(card, 0.7, k, torch.from_numpy(x.reshape(-1)).to(gpu), torch.zeros(rows * card, **i32),
                                   torch.zeros(rows * k, device=gpu), torch.zeros(rows * k, **i32),
                                   g.integers(1, 2**31 - 1, rows).astype(np.uint32), token, score)
    st, got = sampler.sample_temperature_top_k_rows(req, rows, card, card, k)
    assert st == eh.Status.OK, eh.last_error()
    t, s = token.cpu().numpy(), score.cpu().numpy()
    want = [(int(t[r]), float(s[r])) if 0 <= t[r] < card and np.isfinite(s[r]) else eh.Status.INVALID_REQUEST
            for r in range(rows)]
    assert got == want and (rows <= 2 or got[2] == eh.Status.INVALID_REQUEST)
    return got


def test_results_of_growing_batches(gpu):
    s = eh.Sampler()
    for rows in (1, 64, 65, 200, 3):
        sample(gpu, s, rows, rows)


def test_results_into_views(gpu):
    tokens, scores = torch.zeros(40, dtype=torch.int32, device=gpu), torch.zeros(40, device=gpu)
    sample(gpu, eh.Sampler(), 8, 1, tokens[5:13], scores[30:38])


def test_results_from_threads(gpu):
    s = eh.Sampler()
    wrong = []

    def work(seed):
        try:
            for i in range(20):
                sample(gpu, s, 4 + seed, 100 * seed + i)
        except Exception as e:  # handed to the test's thread
            wrong.append(e)

    threads = [threading.Thread(target=work, args=(n,)) for n in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong, wrong
