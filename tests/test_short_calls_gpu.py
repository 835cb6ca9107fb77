"""Calls of a few microseconds, which wait on a word that a small kernel behind them writes: their results are there for any stream
as soon as they return, from every thread, and while other work runs."""
import threading

import numpy as np
import pytest
import torch

import numkong_amd as nk
from tests.test_unaligned_gpu import CALLS, DEV, values_of

pytestmark = pytest.mark.gpu


def calls(count, seed, failures):
    rng = np.random.default_rng(seed)
    elsewhere = torch.cuda.Stream()  # (not ordered behind the library's streams: only the call's return is)
    for number in range(count):
        m, n, k = int(rng.integers(1, 200)), int(rng.integers(1, 3000)), int(rng.integers(1, 300))
        a, b = values_of("i8", m, k, rng).to(DEV), values_of("i8", n, k, rng).to(DEV)
        torch.cuda.current_stream().synchronize()
        got = nk.dots_packed(a, nk.dots_pack(b, "i8"))
        with torch.cuda.stream(elsewhere):
            copy = got.clone()
        elsewhere.synchronize()
        expected = a.cpu().numpy().astype(np.int32) @ b.cpu().numpy().astype(np.int32).T
        if not np.array_equal(copy.cpu().numpy(), expected):
            failures.append((seed, number, m, n, k))


def test_results_are_there_when_the_call_returns():
    failures = []
    calls(60, 101, failures)
    threads = [threading.Thread(target=calls, args=(25, 102 + t, failures)) for t in range(4)]
    for thread in threads:
        thread.start()
    for thread in threads:
        thread.join()
    assert not failures


# A call right behind a long one of another stream's, and one that takes longer than the host looks at the word.
def test_next_to_longer_work():
    rng = np.random.default_rng(110)
    a, b = values_of("i8", 64, 128, rng).to(DEV), values_of("i8", 500, 128, rng).to(DEV)
    packed = nk.dots_pack(b, "i8")
    expected = a.cpu().numpy().astype(np.int32) @ b.cpu().numpy().astype(np.int32).T
    big = torch.randn((4096, 4096), device=DEV)
    for _ in range(5):
        for _ in range(4):
            big = big @ big * 1e-4  # (on the legacy default stream, which the library's streams wait for)
        got = nk.dots_packed(a, packed)
        assert np.array_equal(got.cpu().numpy(), expected)
