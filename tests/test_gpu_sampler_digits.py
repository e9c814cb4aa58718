"""GPU: the sampler's whole-row select where the boundary lies in each of its
four 8-bit digits: fp32 rows whose order keys step by a digit's unit or one less,
positive and negative, against the oracle. The kept set is compared exactly
(top-p where the cut is not within 1e-6 of a cumulative probability).
"""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from oracle import sampler as osm

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("step", [1, 255, 256, 65535, 65536, (1 << 24) - 1])
@pytest.mark.parametrize("V", [61, 9000, 32768])
@pytest.mark.parametrize("negative", [False, True])
def test_boundary_in_each_digit(step, V, negative):
    from tinytron_amd import ops

    n = min(V, (1 << 25) // step)  # distinct steps within the range
    bits = 0x3F800000 + step * (np.random.default_rng(step).permutation(V) % n).astype(np.int64)
    x = bits.astype(np.uint32).view(np.float32).copy()
    x = np.stack([-x if negative else x] * 2)
    for top_k in (65, 200):
        if top_k >= V:
            top_k = V // 2
        _, full = ops.sample_tokens(torch.from_numpy(x).cuda(), top_k=top_k, return_logprobs=True)
        want = osm.filter_logits(x, 1.0, top_k, None)
        assert np.array_equal(np.isfinite(full.cpu().numpy()), np.isfinite(want))
    tok, full = ops.sample_tokens(torch.from_numpy(x).cuda(), top_p=0.5, seed=3, return_logprobs=True)
    full = full.cpu().numpy()
    if osm.top_p_margin(x, 1.0, None, 0.5).min() > 1e-6:
        want = osm.filter_logits(x, 1.0, None, 0.5)
        assert np.array_equal(np.isfinite(full), np.isfinite(want))
    assert np.isfinite(full[[0, 1], tok.cpu().numpy()]).all()
