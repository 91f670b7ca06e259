"""The shared-register wave reductions: every value's sum, exact on integers
(20 values as two Gaussians' nine, 24 as two Gaussians' eleven)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_shared_reductions(hip):
    import torch
    from tinygs_amd import _lib
    vals = np.random.default_rng(3).integers(0, 1000, 64).astype(np.uint32)
    out = torch.zeros(256, dtype=torch.int32, device="cuda")
    inp = torch.from_numpy(vals.view(np.int32)).cuda()
    _lib.check(_lib.load().tgs_selftest_wave(inp.data_ptr(), out.data_ptr(), None))
    torch.cuda.synchronize()
    got = out.cpu().numpy().view(np.float32)
    for start, count in ((192, 24), (216, 20)):
        assert np.array_equal(got[start:start + count], np.float32(vals.sum() + 64 * np.arange(count))), start
    # all 24 (20) values equal
    for start, count in ((68, 24), (92, 20)):
        assert np.array_equal(got[start:start + count], np.full(count, vals.sum(), np.float32)), start
