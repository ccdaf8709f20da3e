"""Per-launch durations: a launch queued behind a running one is timed from
that one's end, a launch on an idle stream from its own start marker, and work
the library does not time never counts."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _step(ctx, a, b, n):
    ctx.call("laplacian", n, n, n, 0.25, 0.125, a, b)


def test_durations_of_queued_and_idle_launches(gpu_ctx):
    n = 256
    a, b = (gpu_ctx.array(np.ones(n ** 3)) for _ in range(2))
    _step(gpu_ctx, a, b, n)
    gpu_ctx.sync()
    gpu_ctx.drain()
    for _ in range(20):            # queued behind each other
        _step(gpu_ctx, a, b, n)
    queued = gpu_ctx.drain()
    for _ in range(20):            # each on an idle stream
        _step(gpu_ctx, a, b, n)
        gpu_ctx.sync()
    idle = gpu_ctx.drain()
    assert len(queued) == len(idle) == 20 and min(queued + idle) > 0
    # the same kernel either way: 16.8 M points take tens of microseconds, a
    # gap counted by mistake would be the host's, or a marker's 4 us
    assert 0.6 < np.median(queued) / np.median(idle) < 1.6


def test_untimed_work_is_not_counted(gpu_ctx, kgmod):
    big = 1 << 27
    x, y = gpu_ctx.empty(big), gpu_ctx.empty(big, np.float32)
    a, b = (gpu_ctx.array(np.ones(32 ** 3)) for _ in range(2))
    for _ in range(2):
        _step(gpu_ctx, a, b, 32)
        gpu_ctx.call("convert", kgmod.F32, y, kgmod.F64, x, big)   # 1.6 GB: over 200 us
        _step(gpu_ctx, a, b, 32)
        gpu_ctx.sync()
        t = gpu_ctx.drain()
    assert len(t) == 2 and max(t) < 150e-6, t


def test_ring_keeps_the_newest_launches(gpu_ctx, kgmod):
    a, b = (gpu_ctx.array(np.ones(8 ** 3)) for _ in range(2))
    gpu_ctx.drain()
    for _ in range(8192 + 7):
        _step(gpu_ctx, a, b, 8)
    t = gpu_ctx.drain(8300)
    assert len(t) == 8192 and min(t) > 0
    gpu_ctx.timing(False)
    try:
        _step(gpu_ctx, a, b, 8)
        gpu_ctx.sync()
        assert gpu_ctx.drain() == []
    finally:
        gpu_ctx.timing(True)
    _step(gpu_ctx, a, b, 8)
    assert len(gpu_ctx.drain()) == 1
