"""How a command is waited for: a wait polls for as long as it is told, then sleeps between its looks."""
import time

import numpy as np
import pytest

import splash_amd
from splash_amd import ops

pytestmark = pytest.mark.gpu


def test_a_caller_chooses_how_long_a_wait_holds_a_core(backend):
    print("case wait", flush=True)
    rows, width = 4096, 4096
    x, y = backend.allocate_buffer(rows * width * 2), backend.allocate_buffer(rows * width * 2)
    weight = backend.from_array(np.full(width, 0x3F80, np.uint16))
    graph = splash_amd.CommandGraph()
    for _ in range(600):   # at least 64 MiB each: not under 10 us
        ops.Normalization.add_rms(graph, x, weight, y, width, rows)
    backend.run(graph)
    share = {}
    try:
        for seconds in (0.0, 10.0):
            backend.set_poll_seconds(seconds)
            ticket = backend.submit_command_async(graph)
            begin, core = time.perf_counter(), time.thread_time()
            ticket.wait()
            share[seconds] = (time.thread_time() - core) / (time.perf_counter() - begin)
    finally:
        backend.set_poll_seconds(0.02)
    print(f"  core held {share[0.0]:.2f} of a wait that sleeps, {share[10.0]:.2f} of one that polls", flush=True)
    assert share[0.0] < 0.5 * share[10.0]
    for seconds in (-1.0, float("nan")):
        with pytest.raises(ValueError):
            backend.set_poll_seconds(seconds)
    backend.run(graph)
