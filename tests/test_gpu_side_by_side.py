"""Planes side by side (fwd_spread) where a launch walks them in several groups, in the float32 kernel too, and in the forms of ragged sizes and of a
rotated walk: every Q tile is the masked softmax of its own plane."""
import pytest
import torch
import torch.nn.functional as F

from sparseattention_amd import compute_mask_kernel, select_tiling, sparse_attention, sparse_attention_tiled, workloads as W

pytestmark = pytest.mark.gpu

TOL = {torch.bfloat16: 2e-2, torch.float16: 4e-3, torch.float32: 1e-5}


def _want(q, k, v, mask):
    wide = torch.float64 if q.dtype == torch.float32 else torch.float32
    o = F.scaled_dot_product_attention(q.to(wide), k.to(wide), v.to(wide), attn_mask=mask)
    return torch.where(mask.any(-1, keepdim=True), o, torch.zeros_like(o))


# K and V of a plane larger than what a group of planes may hold: fours (shared by two XCDs) and eights one after the other, Q tiles that are no
# multiple of two or of four
@pytest.mark.parametrize("H,nQ,D,dtype", [(12, 23, 128, torch.bfloat16), (12, 22, 128, torch.float16), (24, 11, 128, torch.bfloat16), (20, 14, 64, torch.bfloat16),
                                          (12, 23, 64, torch.float32), (24, 11, 64, torch.float32)])
def test_groups_of_planes(gpu, H, nQ, D, dtype):
    Sq, Sk = 64 * nQ, 32768 if (D, dtype) == (64, torch.bfloat16) else 16384
    q, k, v = (torch.randn(1, H, S, D, device=gpu, generator=torch.Generator(device=gpu).manual_seed(S + i)).to(dtype) for i, S in enumerate((Sq, Sk, Sk)))
    g = torch.Generator(device=gpu).manual_seed(H)
    mask = (torch.rand(1, 1, nQ, Sk // 64, device=gpu, generator=g) < 0.05).repeat_interleave(64, 2).repeat_interleave(64, 3)
    mask = mask & (torch.rand(1, 1, Sq, Sk, device=gpu, generator=g) < 0.9)
    mask[..., 40, :] = False
    mask[..., 64 * 5:64 * 6, :] = False  # a tile without entries
    o = sparse_attention(q, k, v, mask.expand(1, H, Sq, Sk), 64, 64)
    assert float((o - _want(q, k, v, mask)).abs().max()) <= TOL[dtype]


@pytest.mark.parametrize("B,H,S,D,BQ,dtype", [(2, 16, 1499, 80, 128, torch.float16), (2, 16, 1100, 120, 128, torch.bfloat16), (3, 12, 1003, 96, 128, torch.bfloat16),
                                              (3, 12, 731, 40, 64, torch.float16), (1, 24, 777, 112, 64, torch.bfloat16)])
def test_ragged_sizes(gpu, B, H, S, D, BQ, dtype):
    assert B * H * (-(-S // BQ)) > 256
    q, k, v = (t[:, :, :S, :D] for t in W.qkv(B, H, S, D, dtype, seed=S, device=gpu))
    i = torch.arange(S, device=gpu)
    mask = torch.stack([(i[None] <= i[:, None]) & (i[None] // (150 + 90 * b) == i[:, None] // (150 + 90 * b)) for b in range(B)])[:, None]
    mask[0, 0, 7] = False
    me = mask.expand(B, H, S, S)
    o = sparse_attention_tiled(q, k, v, select_tiling(me, candidates=((BQ, 64),)))
    assert float((o - _want(q, k, v, me)).abs().max()) <= TOL[dtype]


@pytest.mark.parametrize("B,H,nQ,D", [(2, 12, 14, 128), (3, 12, 9, 64), (1, 20, 15, 128)])
def test_rotated_walk(gpu, B, H, nQ, D):
    S = 128 * nQ
    i = torch.arange(S, device=gpu)
    mask = ((i[None] <= i[:, None]) & (i[:, None] - i[None] < 700)) | (i[None] < 200)
    me = mask[None, None].expand(B, H, S, S)
    q, k, v = W.qkv(B, H, S, D, torch.bfloat16, seed=nQ, device=gpu)
    md = compute_mask_kernel(me, 128, 32)
    o = sparse_attention(q, k, v, me, 128, 32, md, kernel="rotated")
    assert float((o - _want(q, k, v, me)).abs().max()) <= TOL[torch.bfloat16]
