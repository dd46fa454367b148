"""Backward launches whose tiles come by the lengths of their lists: the same bits as in the order of planes, which a workspace without
place for that order gets."""
import math

import pytest
import torch

from sparseattention_amd import _native, compute_backward_metadata, sparse_attention, workloads as W

pytestmark = pytest.mark.gpu


# (D = 64: two passes, D = 128: three; Sq != Sk; lists of one length, which stay as they are)
@pytest.mark.parametrize("D,B,H,Sq,Sk,packed,kind", [
    (64, 4, 12, 2048, 2048, True, "documents"), (64, 1, 124, 512, 512, True, "documents"), (64, 6, 16, 1024, 512, False, "random"),
    (64, 1, 32, 512, 4096, True, "random"), (64, 4, 32, 512, 512, True, "all"), (128, 4, 8, 1024, 1024, True, "documents"),
    (128, 1, 44, 512, 768, False, "random")])
def test_tiles_by_length(gpu, D, B, H, Sq, Sk, packed, kind):
    lib, st = _native.load(), _native.strides
    q, _, _ = W.qkv(B, H, Sq, D, torch.bfloat16, seed=1, device=gpu)
    _, k, v = W.qkv(B, H, Sk, D, torch.bfloat16, seed=2, device=gpu)
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
    lists, packs = [], []
    for md in (bmd.by_query, bmd.by_key):
        for t in (md.unmasked_kv_ids, md.unmasked_lens, md.masked_kv_ids, md.masked_lens):
            lists += [t.data_ptr(), st(t.stride())]
        packs += [md.packed_masks.data_ptr(), st(md.packed_masks.stride()[:2])] if packed else [None, None]
    least, order = lib.sa_bwd_workspace_bytes(B, H, Sq), lib.sa_bwd_order_bytes(B, H, Sq, Sk, D)
    assert order == 4 * B * H * (Sq // 128 + Sk // 128 * (1 if D == 64 else 2))

    def gradients(nbytes, fill):
        out = [torch.full_like(t, float("nan")) for t in (q, k, v)]
        ws = torch.full((least + order + 64,), fill, dtype=torch.uint8, device=gpu)
        tensors = [x for t in (q, k, v, o, do, lse, *out) for x in (t.data_ptr(), st(t.stride()))]
        masks = [None, None, None, None] if packed else [mask.data_ptr(), st(mask.stride()), None, None]
        _native.check(lib.sa_sparse_attention_bwd(*tensors, *masks, *packs, *lists, ws.data_ptr(), nbytes, B, H, Sq, Sk, D,
                                                  _native.SA_DTYPE_BF16, D ** -0.5 / math.log(2), torch.cuda.current_stream().cuda_stream))
        torch.cuda.synchronize()
        assert (ws[nbytes:] == fill).all()
        if nbytes > least:  # every tile has its place
            e = ws[least:least + order].view(torch.int32).view(8, -1).cpu()
            assert all(len(set(row.tolist())) == row.numel() for row in e)
        return out

    want = gradients(least, 0)
    for fill in (0, 255):
        got = gradients(least + order, fill)
        assert all(torch.equal(a, b) for a, b in zip(got, want))
    assert not any(torch.isnan(t).any() for t in want)


def test_what_stays_in_the_order_of_planes():
    f = _native.load().sa_bwd_order_bytes
    assert f(4, 12, 2048, 2048, 64) == 4 * 1536
    assert f(8, 12, 4096, 4096, 64) == 0   # an XCD's planes are more than its L2 holds
    assert f(1, 12, 2048, 2048, 64) == 0   # all tiles run at once
    assert f(1, 61, 1024, 1024, 64) > 0 and f(1, 61, 640, 1152, 64) == 0  # no eighths of one size
    assert f(8, 32, 256, 256, 64) == 0     # lists of four entries at most
    assert f(0, 1, 128, 128, 64) == 0 and f(1, 64, 1000, 1024, 64) == 0 and f(1, 64, 1024, 1024, 96) == 0
