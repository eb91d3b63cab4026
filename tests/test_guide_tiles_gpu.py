"""The training kernel at the edges of its 64-record tiles and of its grid of
one workgroup per CU: gradient and loss against the FP64 oracle that rounds
activations, weights and gradients to bfloat16 where the kernel stores them."""
import ctypes
import time

import numpy as np
import pytest

import guide_oracle as G
from ratbite_amd import _lib as L
from test_guide_gpu import _configure, _params, _records, _set

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 7, 63, 64, 65, 129, 1025, 256 * 64 + 1])
def test_gradient_at_tile_edges(ctx, n):
    _configure(ctx)
    p = _params(5, scale_out=2.0)
    _set(ctx, p)
    rec = _records(n, np.random.default_rng(100 + n))
    # the last record, alone in its tile for most of these sizes, weighs as
    # much as all others together
    rec[-1, 14] = max(float(rec[:-1, 14].sum()), 1.0)
    grad, loss = np.zeros(L.GUIDE_PARAMS, np.float32), ctypes.c_float()
    ctx.check(L.lib().rbh_guide_gradient(ctx.h, L.ptr(rec), n, L.ptr(grad), ctypes.byref(loss)))
    l_ref, g_ref = G.loss_grad(G.unflatten(p.astype(np.float64)), rec.astype(np.float64), emulate_bf16=True)
    ref = G.flatten(g_ref)
    # a value within FP32 rounding of the middle of two bfloat16 values may
    # round the other way: 2^-8 of single terms, and five layers of them
    bound = 5 * 2.0 ** -8
    assert np.linalg.norm(grad - ref) / np.linalg.norm(ref) < bound
    assert abs(loss.value - l_ref) <= 2e-3 * abs(l_ref) + 1e-5
    if n > 1:
        # the bounds tell the last record from a missing or a repeated one
        for wrong in (rec[:-1], np.concatenate([rec[:-1], rec[-2:-1]])):
            l_wrong, g_wrong = G.loss_grad(G.unflatten(p.astype(np.float64)), wrong.astype(np.float64), emulate_bf16=True)
            assert np.linalg.norm(G.flatten(g_wrong) - ref) / np.linalg.norm(ref) > 4 * bound
            assert abs(l_wrong - l_ref) > 2 * (2e-3 * abs(l_ref) + 1e-5)
    # partial sums in a fixed order: the same call gives the same bits
    again = np.zeros_like(grad)
    ctx.check(L.lib().rbh_guide_gradient(ctx.h, L.ptr(rec), n, L.ptr(again), ctypes.byref(loss)))
    assert np.array_equal(grad, again)


def test_large_calls_give_their_memory_back():
    # a million records: 64 MB of input, 164 MB of output; buffers above 128 MiB
    # go with the call
    import ratbite_amd
    rt = ctypes.CDLL("libamdhip64.so")

    def free_bytes():
        free, total = ctypes.c_size_t(), ctypes.c_size_t()
        assert rt.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
        return free.value

    n = 1000003
    rec = np.tile(_records(1, np.random.default_rng(2)), (n, 1))
    out = np.zeros((n, L.GUIDE_OUTPUTS), np.float32)
    with ratbite_amd.Context(0) as c:
        _configure(c)
        # (large enough that the threads of the host copies have their queues)
        c.call("rbh_guide_infer", L.ptr(rec), 50000, L.ptr(out))
        one = out[0].copy()
        free = free_bytes()
        for call in ("rbh_guide_infer", "rbh_guide_infer_fp8", "rbh_guide_infer"):
            c.call(call, L.ptr(rec), n, L.ptr(out))
            # (the driver hands freed memory back a little later)
            end = time.monotonic() + 10.0
            while free - free_bytes() > 130 << 20 and time.monotonic() < end:
                time.sleep(0.05)
            assert free - free_bytes() <= 130 << 20, call
        assert np.array_equal(out[0], one) and np.array_equal(out[-1], one)
