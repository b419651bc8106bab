"""The forward without allocation where the last fp32 row chunk would want more
splits of the vocabulary than its partials have room for in the scratch."""
import pytest
import torch

from mini_trainer_amd import _lib

from test_zz_no_alloc import case, forward_both

pytestmark = pytest.mark.gpu


def test_short_last_chunk_fp32(gpu):
    """Same bound as other fp32 calls, whose split also differs from the
    workspace forward's."""
    T, H, V = 254000, 8, 143753
    X, W, y = case(gpu, T, H, V, torch.float32, 5)
    y[:] = y.clamp(min=0)
    y[177897:] = -100
    assert _lib.load().mt_flce_noalloc_used_bytes(177897, V, 0) <= 16 << 20
    (la, sa), (lb, sb), n = forward_both(gpu, X, W, y, 0.0)
    assert n == 177897
    assert not torch.isnan(lb).any() and not torch.isnan(sb).any()
    assert float(((la - lb).abs() / la.abs().clamp(min=1e-3)).max()) <= 1e-6
    assert float(((sa - sb).abs() / sa.abs()).max()) <= 1e-6
