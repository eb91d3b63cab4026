"""The training kernel at the edges of its 64-record tiles and of its grid of
one workgroup per CU: gradient and loss against the FP64 oracle that rounds
activations, weights and gradients to bfloat16 where the kernel stores them."""
import ctypes

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
    grad, loss = np.zeros(L.GUIDE_PARAMS, np.float32), ctypes.c_float()
    ctx.check(L.lib().rbh_guide_gradient(ctx.h, L.ptr(rec), n, L.ptr(grad), ctypes.byref(loss)))
    l_ref, g_ref = G.loss_grad(G.unflatten(p.astype(np.float64)), rec.astype(np.float64), emulate_bf16=True)
    ref = G.flatten(g_ref)
    # a value within FP32 rounding of the middle of two bfloat16 values may
    # round the other way: 2^-8 of single terms, and five layers of them
    assert np.linalg.norm(grad - ref) / np.linalg.norm(ref) < 5 * 2.0 ** -8
    assert abs(loss.value - l_ref) <= 2e-3 * abs(l_ref) + 1e-5
    # partial sums in a fixed order: the same call gives the same bits
    again = np.zeros_like(grad)
    ctx.check(L.lib().rbh_guide_gradient(ctx.h, L.ptr(rec), n, L.ptr(again), ctypes.byref(loss)))
    assert np.array_equal(grad, again)
