"""Backward launches whose tiles come by the lengths of their lists: the same bits as in the order of planes, which a workspace without
place for that order gets."""
import math

import pytest
import torch

from sparseattention_amd import _native, compute_backward_metadata, sparse_attention, workloads as W

pytestmark = pytest.mark.gpu


def backward(gpu, D, B, H, Sq, Sk, packed, kind, dtype):
    """gradients(bytes of workspace, what it holds before) -> the gradients and the workspace behind the statistics"""
    lib, st = _native.load(), _native.strides
    q, _, _ = W.qkv(B, H, Sq, D, dtype, seed=1, device=gpu)
    _, k, v = W.qkv(B, H, Sk, D, dtype, seed=2, device=gpu)
    do = torch.randn_like(q)
    g = torch.Generator(device=gpu).manual_seed(D + H)
    if kind == "documents":
        ids = (torch.rand(B, Sk, device=gpu, generator=g) < 1 / 300).cumsum(1)
        mask = (ids[:, :Sq, None] == ids[:, None, :]) & (torch.arange(Sk, device=gpu)[None, None] <= torch.arange(Sq, device=gpu)[None, :, None])
    elif kind == "random":  # (lists of all lengths, empty ones among them)
        tiles = torch.rand(B, Sq // 64, Sk // 64, device=gpu, generator=g) < torch.rand(B, Sq // 64, 1, device=gpu, generator=g)
        mask = tiles.repeat_interleave(64, 1).repeat_interleave(64, 2) & (torch.rand(B, Sq, Sk, device=gpu, generator=g) < 0.9)
    else:
        mask = torch.ones(B, Sq, Sk, dtype=torch.bool, device=gpu)
    mask = mask[:, None].expand(B, H, Sq, Sk)
    o, lse = sparse_attention(q, k, v, mask, 128, 64, return_lse=True)
    bmd = compute_backward_metadata(mask, pack_partial=packed)
    least, order = lib.sa_bwd_workspace_bytes(B, H, Sq), lib.sa_bwd_order_bytes(B, H, Sq, Sk, D)
    assert order == 4 * B * H * (Sq // 128 + Sk // 128 * (1 if D == 64 else 2))

    def gradients(with_order, fill):
        nbytes = least + (order if with_order else 0)
        out = [torch.full_like(t, float("nan")) for t in (q, k, v)]
        lists, packs = [], []
        for md in (bmd.by_query, bmd.by_key):
            for t in (md.unmasked_kv_ids, md.unmasked_lens, md.masked_kv_ids, md.masked_lens):
                lists += [t.data_ptr(), st(t.stride())]
            packs += [md.packed_masks.data_ptr(), st(md.packed_masks.stride()[:2])] if packed else [None, None]
        ws = torch.full((least + order + 64,), fill, dtype=torch.uint8, device=gpu)
        tensors = [x for t in (q, k, v, o, do, lse, *out) for x in (t.data_ptr(), st(t.stride()))]
        masks = [None, None, None, None] if packed else [mask.data_ptr(), st(mask.stride()), None, None]
        _native.check(lib.sa_sparse_attention_bwd(*tensors, *masks, *packs, *lists, ws.data_ptr(), nbytes, B, H, Sq, Sk, D,
                                                  _native.SA_DTYPE_BF16 if dtype == torch.bfloat16 else _native.SA_DTYPE_FP16,
                                                  D ** -0.5 / math.log(2), torch.cuda.current_stream().cuda_stream))
        torch.cuda.synchronize()
        assert (ws[nbytes:] == fill).all()
        return out, ws[least:nbytes]
    return gradients


# (D = 64: two passes, D = 128: three; Sq != Sk; lists of one length, which stay as they are)
@pytest.mark.parametrize("D,B,H,Sq,Sk,packed,kind,dtype", [
    (64, 4, 12, 2048, 2048, True, "documents", torch.bfloat16), (64, 1, 124, 512, 512, True, "documents", torch.bfloat16),
    (64, 6, 16, 1024, 512, False, "random", torch.bfloat16), (64, 3, 32, 512, 1024, True, "random", torch.bfloat16),
    (64, 4, 32, 512, 512, True, "all", torch.bfloat16), (64, 4, 32, 512, 512, True, "documents", torch.float16),
    (64, 1, 128, 512, 512, False, "random", torch.float16), (128, 4, 8, 1024, 1024, True, "documents", torch.bfloat16),
    (128, 1, 32, 1024, 1280, False, "random", torch.bfloat16), (128, 1, 32, 1024, 1024, True, "random", torch.float16),
    (128, 2, 8, 2048, 2048, False, "documents", torch.float16), (64, 2, 12, 4096, 4096, False, "documents", torch.bfloat16)])
def test_tiles_by_length(gpu, D, B, H, Sq, Sk, packed, kind, dtype):
    gradients = backward(gpu, D, B, H, Sq, Sk, packed, kind, dtype)
    want, _ = gradients(False, 0)
    for fill in (0, 255):
        got, order = gradients(True, fill)
        assert all(torch.equal(a, b) for a, b in zip(got, want))
        e = order.view(torch.int32).view(8, -1).cpu()  # every tile has its place
        assert all(len(set(row.tolist())) == row.numel() for row in e)
    assert not any(torch.isnan(t).any() for t in want)


def test_what_stays_in_the_order_of_planes():
    f = _native.load().sa_bwd_order_bytes
    assert f(4, 12, 2048, 2048, 64) == 4 * 1536
    assert f(8, 12, 4096, 4096, 64) == 0   # an XCD's planes are more than its L2 holds
    assert f(1, 12, 2048, 2048, 64) == 0   # all tiles run at once
    assert f(1, 61, 1024, 1024, 64) > 0 and f(1, 61, 640, 1152, 64) == 0  # no eighths of one size
    assert f(8, 32, 256, 256, 64) == 0     # lists of four entries at most
    assert f(2, 8, 2048, 2048, 128) > 0 and f(1, 64, 512, 512, 128) == 0  # D = 128: of eight at most
    assert f(1, 8, 8192, 8192, 64) == 0 and f(1, 8, 4096, 4096, 128) == 0  # a XCD has one plane
    assert f(2, 12, 4096, 4096, 64) > 0 and f(2, 8, 4096, 4096, 64) == 0 and f(1, 16, 3072, 3072, 128) > 0  # two long ones
    assert f(1, 48, 1024, 4096, 64) > 0 and f(1, 32, 512, 4096, 64) == 0  # the sort takes longer than the statistics
    assert f(0, 1, 128, 128, 64) == 0 and f(1, 64, 1000, 1024, 64) == 0 and f(1, 64, 1024, 1024, 96) == 0
