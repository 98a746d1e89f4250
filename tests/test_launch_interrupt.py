"""Runs of steps enqueued natively stay under the caller's control (host-only launch lists: parity
swaps, no GPU)."""
import signal
import time
from types import SimpleNamespace

import pytest

from virtualfluids_amd import capi
from virtualfluids_amd.launches import LaunchList

STREAM = SimpleNamespace(cuda_stream=0)


def _swaps(n):
    p = capi.LBMParameter()
    p.isEvenTimestep = 1
    out = LaunchList()
    for _ in range(n):
        out.swap(p)
    return p, out


def test_a_long_run_answers_a_signal():
    """The list of this run takes minutes; a signal after 0.2 s ends it."""
    _, out = _swaps(200)

    class Interrupted(Exception):
        pass

    def handler(signum, frame):
        raise Interrupted

    old = signal.signal(signal.SIGALRM, handler)
    start = time.monotonic()
    try:
        signal.setitimer(signal.ITIMER_REAL, 0.2)
        with pytest.raises(Interrupted):
            out.run(1 << 24, STREAM)
    finally:
        signal.setitimer(signal.ITIMER_REAL, 0)
        signal.signal(signal.SIGALRM, old)
    assert time.monotonic() - start < 2.0


@pytest.mark.parametrize("n", [0, 1, 255, 256, 257, 1000])
def test_every_repeat_is_enqueued(n):
    p, out = _swaps(3)
    out.run(n, STREAM)
    assert p.isEvenTimestep == (1 + 3 * n) % 2


@pytest.mark.parametrize("n", [4.0, 3.5, 300.0, "int64", "float64"])
def test_step_counts_need_not_be_ints(n):
    """A count of steps computed from times (T / dt) runs until it is used up."""
    import math

    import numpy as np

    n = {"int64": np.int64(300), "float64": np.float64(299.5)}.get(n, n)
    p, out = _swaps(1)
    out.run(n, STREAM)
    assert p.isEvenTimestep == (1 + math.ceil(n)) % 2
