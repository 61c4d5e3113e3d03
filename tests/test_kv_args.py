"""The addresses and strides that the decode takes of a cache are those of its
K and V views, in every cache layout."""
import pytest
import torch

from locks.attention.decode import _kv_args, _split_kv


@pytest.mark.parametrize("shape", [
    (5, 2, 16, 3, 8), (2, 5, 16, 3, 8), (2, 2, 16, 3, 8), (2, 1, 16, 3, 8), (1, 2, 16, 1, 8), (5, 1, 16, 3, 8),
    (1, 1, 16, 3, 8)])
@pytest.mark.parametrize("heads_first", [False, True])
def test_equal_the_views(shape, heads_first):
    kv = torch.arange(1 + torch.Size(shape).numel(), dtype=torch.int16).view(torch.bfloat16)[1:].view(shape)
    if heads_first:                                   # heads ahead of tokens in memory
        kv = kv.transpose(2, 3).contiguous().transpose(2, 3)
    k, v = _split_kv(kv)
    kp, vp, strides, dims = _kv_args(kv)
    assert kp == k.data_ptr() and strides == k.stride()[:3] and dims == tuple(k.shape)
    if v is None:
        assert vp is None
    else:
        assert vp == v.data_ptr() and strides == v.stride()[:3] and dims == tuple(v.shape)


def test_k_only_cache_needs_a_tier():
    from locks.attention import decode as D

    class St:
        n_kv, b_max, sink_pages, window_pages = 3, 4, 1, 1

    with pytest.raises(ValueError, match="K-only"):
        D.sparse_paged_decode_batched(torch.zeros(1, 3, 8), torch.zeros(5, 1, 16, 3, 8), None,
                                      torch.zeros(1, dtype=torch.int32), St, torch.zeros(1, 3, 8), scale=1.0)
