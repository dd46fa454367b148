"""Decode whose K comes as whole rows and crosses the lanes through LDS (calls with lists), against the launch that makes its
lists itself and reads K per lane: the same operands reach the same products in the same order, so outputs are equal bit for bit."""
import pytest
import torch

from sparseattention_amd import compute_mask_kernel, sparse_attention_decode, workloads as W

pytestmark = pytest.mark.gpu


# (one chunk per workgroup and fewer than waves; rows of another stride than their length; both element types and head dims)
@pytest.mark.parametrize("dtype,D", [(torch.bfloat16, 128), (torch.float16, 128), (torch.bfloat16, 64), (torch.float16, 64)])
@pytest.mark.parametrize("Sq,Sk,BK,splits", [(1, 32, 32, 1), (1, 512, 32, 4), (7, 1024, 64, 3), (32, 1024, 256, 2), (2, 8192, 128, 1)])
@pytest.mark.parametrize("layout", ["bhsd", "bshd", "rows apart"])
def test_key_rows_as_keys_per_lane(gpu, dtype, D, Sq, Sk, BK, splits, layout):
    B, H = 2, 3
    q, k, v = W.qkv(B, H, Sq, D, dtype, seed=Sk + D, device=gpu, Sk=Sk)
    if layout == "bshd":
        k, v = (t.transpose(1, 2).contiguous().transpose(1, 2) for t in (k, v))
    elif layout == "rows apart":
        wide = torch.full((B, H, Sk, D + 24), float("nan"), dtype=dtype, device=gpu)  # (nothing between the rows may be read)
        wide[..., :D] = k
        k = wide[..., :D]
    g = torch.Generator().manual_seed(Sk)
    mask = torch.rand(B, 1, Sq, Sk, generator=g) < 0.7
    mask[..., : Sk // 2] = True
    mask = mask.to(gpu).expand(B, H, Sq, Sk)
    md = compute_mask_kernel(mask, Sq, BK)
    by_rows = sparse_attention_decode(q, k, v, mask, BK, md, num_splits=splits)
    per_lane = sparse_attention_decode(q, k, v, mask, BK, num_splits=splits)
    assert not torch.isnan(by_rows).any()
    assert torch.equal(by_rows, per_lane)
