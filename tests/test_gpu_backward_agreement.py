"""Backward metadata whose two lists do not say the same: dQ follows by_query, dK and dV by_key, also at the sizes where lists
of one mask take the passes that store dS."""
import copy

import pytest
import torch

from sparseattention_amd import _native, compute_backward_metadata, sparse_attention, sparse_attention_backward, workloads as W
from sparseattention_amd.sparse_attn_kernel import BackwardMetadata

pytestmark = pytest.mark.gpu
B, H, S, D = 1, 64, 1024, 128


def _inputs(gpu):
    q, k, v = W.qkv(B, H, S, D, torch.bfloat16, seed=5, device=gpu)
    mask = torch.ones(S, S, dtype=torch.bool, device=gpu).tril()[None, None].expand(B, H, S, S)
    o, lse = sparse_attention(q, k, v, mask, 128, 64, return_lse=True)
    return torch.randn_like(q), q, k, v, o, lse, mask


def _poison(gpu):
    """Leaves NaN patterns in the memory that the next workspace is taken from."""
    torch.full((_native.load().sa_bwd_workspace_bytes_ex(B, H, S, S, D),), 0xFF, dtype=torch.uint8, device=gpu)


def test_key_lists_of_fewer_keys(gpu):
    assert _native.load().sa_bwd_workspace_bytes_ex(B, H, S, S, D) > _native.load().sa_bwd_workspace_bytes(B, H, S)
    do, q, k, v, o, lse, mask = _inputs(gpu)
    first = mask.clone()
    first[..., S // 2:] = False  # gradients of the first half of the keys only
    whole, part = compute_backward_metadata(mask), compute_backward_metadata(first)
    _poison(gpu)
    dq, dk, dv = sparse_attention_backward(do, q, k, v, o, lse, None, BackwardMetadata(whole.by_query, part.by_key))
    want = sparse_attention_backward(do, q, k, v, o, lse, None, whole)
    for got, w in ((dq, want[0]), (dk[:, :, : S // 2], want[1][:, :, : S // 2]), (dv[:, :, : S // 2], want[2][:, :, : S // 2])):
        # both within 3.2e-3 of float64
        assert float((got.double() - w.double()).norm() / w.double().norm()) <= 6.4e-3
    assert not dk[:, :, S // 2:].any() and not dv[:, :, S // 2:].any()


@pytest.mark.parametrize("how", ["replaced", "edited", "copied"])
def test_lists_changed_later(gpu, how):
    """What was known of lists of one mask is void with the lists: the same gradients as from lists put together anew."""
    do, q, k, v, o, lse, mask = _inputs(gpu)
    bmd = compute_backward_metadata(mask)
    if how == "replaced":
        first = mask.clone()
        first[..., S // 2:] = False
        bmd.by_key = compute_backward_metadata(first).by_key
    elif how == "edited":
        bmd.by_key.unmasked_lens.zero_()
    else:
        bmd = copy.deepcopy(bmd)
        assert bmd._agreeing is None
    _poison(gpu)
    got = sparse_attention_backward(do, q, k, v, o, lse, None, bmd)
    want = sparse_attention_backward(do, q, k, v, o, lse, None, BackwardMetadata(bmd.by_query, bmd.by_key))
    assert all(torch.isfinite(x).all() and torch.equal(x, y) for x, y in zip(got, want))


def test_lists_of_one_mask_with_a_transposed_mask_beside_them(gpu):
    """The packed tiles are what is read, as without it; a transposed mask of other sizes is refused as ever."""
    do, q, k, v, o, lse, mask = _inputs(gpu)
    bmd = compute_backward_metadata(mask)
    want = sparse_attention_backward(do, q, k, v, o, lse, None, bmd)
    bmd.transposed_mask = mask.transpose(-1, -2).contiguous()
    got = sparse_attention_backward(do, q, k, v, o, lse, None, bmd)
    assert all(torch.equal(x, y) for x, y in zip(got, want))
    bmd.transposed_mask = mask[..., :128]
    with pytest.raises(ValueError):
        sparse_attention_backward(do, q, k, v, o, lse, None, bmd)
