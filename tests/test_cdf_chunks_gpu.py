"""Env-map tables where a row's chunks begin and end: 1024 lanes of four texels
a chunk, one or two chunks kept in registers, more through LDS."""
import numpy as np
import pytest

import oracle_lib as O
from ratbite_amd.envmaps import lognormal_envmap

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("channels", [3, 4])
@pytest.mark.parametrize("w,h", [(64, 32), (1028, 16), (2052, 12), (4096, 8), (4100, 8), (8188, 8), (8192, 4), (8196, 4),
                                 (16388, 4)])
def test_rows_at_chunk_edges(ctx, w, h, channels):
    tex = lognormal_envmap(w, h, sigma=2.0, seed=w + h, sun=True)
    tex[h // 2] = 0.0
    given = tex if channels == 3 else np.ascontiguousarray(np.concatenate([tex, np.ones((h, w, 1), np.float32)], axis=2))
    ctx.envmap_build(given)
    cond, marg, cdfy, _ = ctx.envmap_read()
    ocx, ocy, _ = O.cdf_build(tex)
    ocond, omarg = O.cdf_invert(ocx, ocy)
    assert np.array_equal(cond, ocond) and np.array_equal(marg, omarg) and np.array_equal(cdfy, ocy)
    ctx.envmap_build(given, fp64=True)
    cond, marg, cdfy, integral = ctx.envmap_read()
    dx, dy, dint = O.cdf_build_f64(tex)
    # one rounding of a double per value (sums of at most 2^14 doubles: 2^-39)
    assert np.max(np.abs(cdfy.astype(np.float64) - dy)) <= 2.0 ** -24
    assert abs(integral - dint / (w * h)) / (dint / (w * h)) < 1e-12
    ocond, _ = O.cdf_invert(dx.astype(np.float32), dy.astype(np.float32))
    diff = np.abs(cond.astype(np.int64) - ocond.astype(np.int64))
    assert diff.max() <= 1 and np.mean(diff == 0) > 0.999
