"""Decode on a small mask without lists (sa_sparse_attention_decode_mask): bit for bit what the path over lists gives."""
import ctypes

import pytest
import torch

from sparseattention_amd import _native, compute_mask_kernel, sparse_attention_decode, workloads as W


def fits(ptr, strides, B, H, Sq, Sk, BK):
    return _native.load().sa_decode_mask_fits(ptr, _native.strides(strides), B, H, Sq, Sk, BK)


def test_rule_of_the_direct_path():
    p = ctypes.c_void_p(1 << 20)
    assert fits(p, (0, 0, 2048, 1), 4, 32, 1, 2048, 64)
    assert fits(p, (32768, 0, 1024, 1), 4, 32, 32, 1024, 256) and fits(p, (0, 0, 0, 1), 4, 32, 1, 32768, 32)
    assert fits(p, (7, 7, 7, 1), 1, 1, 1, 32, 32)  # (strides of dimensions of size 1 are never used)
    assert not fits(p, (0, 0, 2048, 1), 4, 32, 17, 2048, 64) and not fits(p, (0, 0, 0, 1), 1, 1, 1, 32800, 32)
    assert not fits(p, (0, 0, 64, 1), 1, 1, 33, 64, 32) and not fits(p, (0, 0, 64, 1), 1, 1, 1, 64, 16)
    assert not fits(p, (0, 0, 0, 1), 1, 1, 1, 96, 48) and not fits(p, (0, 0, 0, 1), 1, 1, 1, 512, 512)
    assert not fits(p, (0, 0, 96, 1), 1, 1, 1, 96, 64) and not fits(p, (0, 0, 0, 1), 1, 1, 1, 64, 0)
    assert not fits(p, (0, 0, 2, 2), 1, 1, 1, 64, 32) and not fits(p, (0, 0, 0, 0), 1, 1, 1, 64, 32)
    for i in range(3):
        s = [64, 64, 64, 1]
        s[i] = 72
        assert not fits(p, s, 2, 2, 2, 64, 32)
    assert not fits(ctypes.c_void_p((1 << 20) + 8), (0, 0, 64, 1), 1, 1, 1, 64, 32) and not fits(None, (0, 0, 64, 1), 1, 1, 1, 64, 32)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("Sq,Sk,D,BK,form", [(1, 32, 64, 32, "own"), (1, 32768, 128, 64, "heads"), (32, 1024, 64, 32, "own"),
                                            (16, 2048, 128, 128, "heads"), (3, 1088, 128, 64, "planes"), (31, 1024, 128, 256, "rows"),
                                            (2, 2080, 128, 32, "offset"), (5, 544, 80, 32, "bytes")])
def test_same_as_with_lists(gpu, Sq, Sk, D, BK, form, dtype):
    B, H = 2, 3
    q, k, v = W.qkv(B, H, Sq, D, dtype, seed=Sq + Sk, device=gpu, Sk=Sk)
    g = torch.Generator().manual_seed(Sk + Sq)
    lead = {"own": (B, H), "heads": (B, 1), "planes": (1, 1)}.get(form, (B, H))
    kind = torch.randint(0, 3, (*lead, 1, Sk // 16), generator=g).repeat_interleave(16, -1)
    kind[..., Sk // 2:] = 0  # the second half empty: workgroups and waves without a chunk
    m = (kind == 2) | ((kind == 1) & (torch.rand(*lead, Sq, Sk, generator=g) < 0.5))
    m = m.to(gpu)
    if Sq > 2:
        m[:, :, 1] = False  # a row without a key
    m[:, :, 0, 0] = True
    if form == "rows":
        m = m[:, :, :1]
    if form == "offset":  # a window into a larger tensor
        big = torch.ones(B, H, Sq + 1, Sk + 32, dtype=torch.bool, device=gpu)
        big[:, :, 1:, 16:-16] = m
        m = big[:, :, 1:, 16:-16]
    if form == "bytes":  # any byte but 0 attends
        m = (m.to(torch.uint8) * torch.randint(1, 256, m.shape, generator=g, dtype=torch.uint8).to(gpu)).view(torch.bool)
    mask = m.expand(B, H, Sq, Sk)
    assert fits(mask.data_ptr(), mask.stride(), B, H, Sq, Sk, BK)
    ones = mask.view(torch.uint8) != 0
    md = compute_mask_kernel(ones, Sq, BK)
    empty = Sk // 2 + BK  # from here on no row attends: never read
    k[:, :, empty:], v[:, :, empty:] = float("nan"), float("nan")
    for splits in (0, 1, 7):
        want, wlse = sparse_attention_decode(q, k, v, ones, BK, md, num_splits=splits, return_lse=True)
        o, lse = sparse_attention_decode(q, k, v, mask, BK, num_splits=splits, return_lse=True)
        torch.cuda.synchronize()
        assert not torch.isnan(o).any() and torch.equal(o, want) and torch.equal(lse, wlse)
