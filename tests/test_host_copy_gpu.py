"""Host copies around the sizes where they go from the runtime to the threads
(2 MiB) and change their chunks, from several threads at once, and from
pinned memory: every byte comes back."""
import threading

import numpy as np
import pytest
import torch

import ratbite_amd
from ratbite_amd import _lib as L

pytestmark = pytest.mark.gpu


def _round_trip(ctx, w, h, seed, accum=None):
    a = np.random.default_rng(seed).standard_normal((h, w, 4)) if accum is None else accum
    b = np.zeros_like(a)
    ctx.call("rbh_write_accum", L.ptr(a), w, h)
    ctx.call("rbh_read_accum", L.ptr(b))
    assert np.array_equal(a, b)


# 32 bytes a pixel: 2 MiB is 65536 of them, a full chunk of every thread 262144
@pytest.mark.parametrize("pixels", [1, 65535, 65536, 65537, 131071, 262144, 262145, 1000003])
def test_round_trip(ctx, pixels):
    _round_trip(ctx, pixels, 1, pixels)


def test_threads_share_the_pool():
    errors = []

    def body(seed):
        try:
            with ratbite_amd.Context(0) as c:
                for i in range(4):
                    _round_trip(c, 70000 + 1000 * seed + i, 3, seed)
        except BaseException as e:   # noqa: BLE001 - reported by the test
            errors.append(e)

    ts = [threading.Thread(target=body, args=(k,)) for k in range(4)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not errors


def test_pinned_memory(ctx):
    t = torch.randn((256, 512, 4), dtype=torch.float64, generator=torch.Generator().manual_seed(3)).pin_memory()
    _round_trip(ctx, 512, 256, 0, accum=t.numpy())
