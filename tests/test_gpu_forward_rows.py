"""The preprocess's staged SH rows: colours (through the forward's bit-exact
check) for primitive counts around the staged parts' edges and the last whole
16 bytes of a run, at each storage type and rasterizer."""
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
