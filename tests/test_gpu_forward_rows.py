"""The preprocess's staged SH rows and the rect walks, through the forward's
bit-exact check: primitive counts around the staged parts' edges and the last
whole 16 bytes of a run, and rects of every size, in each rasterizer."""
import dataclasses

import numpy as np
import pytest

from tinygs_amd import scenes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sh_dtype", ["float32", "float16"])
@pytest.mark.parametrize("n", [1, 127, 129, 255, 257, 385])
def test_colors_by_count(hip, orc, n, sh_dtype):
    from test_gpu_fgs16 import _check_forward as check16, _render16
    from test_gpu_parity import _check_forward
    s = scenes.config2(seed=17, n=n, width=131, height=77)
    s = dataclasses.replace(s, sh_degree=1 + n % 3, scales=s.scales + np.float32(1.0), sh_dtype=sh_dtype,
                            sh0=s.sh0.astype(np.float16).astype(np.float32),
                            sh_rest=s.sh_rest.astype(np.float16).astype(np.float32))
    _check_forward(s, orc)
    check16(s, orc, _render16(s))


def test_rects_by_size(hip, orc):
    """Tile counts and instances of rects from one tile to the whole grid (132 x 19 tiles, wider than a wave), the
    small and the big ones in the same waves."""
    from test_gpu_fgs16 import _check_forward as check16, _render16
    from test_gpu_parity import _check_forward
    s = scenes.config2(seed=19, n=600, width=2100, height=300)
    scales = (np.linspace(-5.5, 0.3, 600, dtype=np.float32)[np.random.default_rng(2).permutation(600), None]
              + 0.7 * (s.scales + 4.0)).astype(np.float32)
    s = dataclasses.replace(s, scales=scales)
    run, (pre, bins, fwd) = _check_forward(s, orc)
    b = pre["bounds"].reshape(-1, 4)[pre["n_touched"] > 0].astype(np.int64)
    rect = (b[:, 1] - b[:, 0]) * (b[:, 3] - b[:, 2])
    assert (rect <= 8).any() and ((rect > 32) & (rect <= 64)).any() and (rect > 1000).any()
    check16(s, orc, _render16(s))
