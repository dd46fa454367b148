"""Forward launches with too few Q tiles to fill the device: lists shared by several workgroups and merged."""
import pytest
import torch

from sparseattention_amd import MaskMetadata, _native, compute_mask_kernel, sparse_attention, workloads as W

pytestmark = pytest.mark.gpu

TOL = {torch.bfloat16: 2e-2, torch.float16: 4e-3, torch.float32: 1e-5}


@pytest.mark.parametrize("dtype,B,H,Sq,Sk,D,BQ,BK", [
    (torch.bfloat16, 1, 3, 256, 4096, 128, 128, 64),   # three planes: the last pair of planes is half empty
    (torch.bfloat16, 1, 1, 128, 2048, 128, 128, 32),   # one Q tile, the shortest rows that are shared
    (torch.bfloat16, 2, 1, 192, 2112, 64, 64, 16),     # four entries per chunk, rows that end in part of a chunk
    (torch.float16, 1, 2, 96, 8192, 128, 32, 256),     # entries of several chunks
    (torch.bfloat16, 1, 1, 64, 4096, 64, 64, 2048),    # fewer entries than parts
    (torch.bfloat16, 5, 5, 640, 3072, 128, 128, 64),   # 125 tiles: parts of 16 chunks
    (torch.float32, 1, 3, 192, 1056, 64, 64, 32),
    (torch.float32, 1, 2, 256, 512, 128, 128, 16),
    (torch.float32, 2, 1, 64, 4096, 64, 32, 1024),
])
@pytest.mark.parametrize("packed", [True, False])
def test_shared_lists(gpu, dtype, B, H, Sq, Sk, D, BQ, BK, packed):
    g = torch.Generator().manual_seed(Sk + D)
    q, _, _ = W.qkv(B, H, Sq, D, dtype, seed=1, device=gpu)
    _, k, v = W.qkv(B, H, Sk, D, dtype, seed=2, device=gpu)
    mask = torch.rand(B, 1, Sq, Sk, generator=g) < 0.5
    step = 32 if BK < 64 else 64
    for c in range(0, Sk, 4 * step):  # runs of FULL, PARTIAL and EMPTY tiles, in no order that parts could follow
        mask[..., c:c + step] = True
        mask[..., c + step:c + 2 * step] = False
    mask[:, :, : BQ, : Sk // 3] = True
    mask[0, 0, 5] = False           # a row that attends to nothing
    mask[0, 0, 7, Sk // 4:] = False  # and one whose keys all lie in the first parts
    if Sq > BQ:
        mask[-1, 0, BQ:2 * BQ, 300:] = False  # a tile whose list is too short to be shared
    mask = mask.to(gpu).expand(B, H, Sq, Sk)
    assert _native.load().sa_fwd_split_workspace_bytes(B, H, Sq, Sk, D, BQ, BK, {torch.bfloat16: 0, torch.float16: 1}.get(dtype, 2)) > 0
    md = compute_mask_kernel(mask, BQ, BK, pack_partial=packed)
    o, lse = sparse_attention(q, k, v, mask, BQ, BK, mask_metadata=md, return_lse=True)
    again = sparse_attention(q, k, v, mask, BQ, BK, mask_metadata=md)
    assert torch.equal(o, again)
    s = (q.double() @ k.double().transpose(-1, -2).contiguous()) * D ** -0.5
    s = s.masked_fill(~mask, float("-inf"))
    want_lse = torch.logsumexp(s, -1)
    want = torch.nan_to_num(torch.softmax(s, -1)) @ v.double()
    assert float((o.double() - want).abs().max()) <= TOL[dtype]
    live = torch.isfinite(want_lse)
    assert torch.equal(torch.isfinite(lse), live) and not live[0, 0, 5].any()
    assert float((lse.double() - want_lse)[live].abs().max()) <= (1e-5 if dtype == torch.float32 else 6e-3 + 2 ** -9 * 5)
    assert torch.equal(o[0, :, 5], torch.zeros_like(o[0, :, 5]))


def test_caller_lists_are_clamped_in_shared_lists(gpu):
    """Counts beyond the row and indices outside it read nothing outside K, V and the packed tiles (values: the clean
    entries alone)."""
    B, H, Sq, Sk, D, BQ, BK = 1, 2, 128, 2048, 128, 128, 64
    q, _, _ = W.qkv(B, H, Sq, D, torch.bfloat16, seed=3, device=gpu)
    _, k, v = W.qkv(B, H, Sk, D, torch.bfloat16, seed=4, device=gpu)
    mask = torch.ones(B, H, Sq, Sk, dtype=torch.bool, device=gpu)
    md = compute_mask_kernel(mask, BQ, BK)
    ids = md.unmasked_kv_ids.clone()
    ids[..., 3], ids[..., 20] = Sk // BK, -1
    bad = MaskMetadata(ids, md.unmasked_lens.clone(), md.masked_kv_ids, md.masked_lens, md.packed_masks)
    from sparseattention_amd.mask_utils import validation_key
    bad._validated_for = validation_key(bad, Sk, BK)  # (past the wrapper's own check)
    got = sparse_attention(q, k, v, mask, BQ, BK, mask_metadata=bad)
    clean = mask.clone()
    clean[..., 3 * BK:4 * BK] = False
    clean[..., 20 * BK:21 * BK] = False
    want = torch.nn.functional.scaled_dot_product_attention(q.float(), k.float(), v.float(), attn_mask=clean)
    assert float((got.float() - want).abs().max()) <= 2e-2


@pytest.mark.parametrize("tiles,chunks", [(65, 16), (96, 20), (128, 17), (128, 24)])
def test_lists_too_short_to_be_shared(gpu, tiles, chunks):
    """Half the device's slots taken: two workgroups beside each other are no faster on such a list than one (results as
    of one, bit for bit)."""
    B, H, D, BQ, BK, Sk = 1, 1, 128, 128, 64, 8192
    q, _, _ = W.qkv(B, H, BQ * tiles, D, torch.bfloat16, seed=3, device=gpu)
    _, k, v = W.qkv(B, H, Sk, D, torch.bfloat16, seed=4, device=gpu)
    mask = (torch.arange(Sk, device=gpu) >= Sk - BK * chunks).expand(B, H, BQ * tiles, Sk)
    md = compute_mask_kernel(mask, BQ, BK)
    assert _native.load().sa_fwd_split_workspace_bytes(B, H, BQ * tiles, Sk, D, BQ, BK, 0) > 0
    got = sparse_attention(q, k, v, None, BQ, BK, md)
    many = torch.cat([q] * 4, 2)  # (enough Q tiles to fill the device: nothing is shared)
    more = compute_mask_kernel(mask[:, :, :1].expand(B, H, 4 * BQ * tiles, Sk), BQ, BK)
    assert torch.equal(got, sparse_attention(many, k, v, None, BQ, BK, more)[:, :, :BQ * tiles])


@pytest.mark.parametrize("keys", [512, 576])
def test_no_parts_where_the_metadata_says_that_no_list_is_long(gpu, keys):
    B, H, Sq, Sk, D, BQ, BK = 1, 4, 128, 8192, 64, 128, 64
    q, _, _ = W.qkv(B, H, Sq, D, torch.bfloat16, seed=3, device=gpu)
    _, k, v = W.qkv(B, H, Sk, D, torch.bfloat16, seed=4, device=gpu)
    mask = (torch.arange(Sk, device=gpu) >= Sk - keys).expand(B, H, Sq, Sk)
    md = compute_mask_kernel(mask, BQ, BK)
    want = sparse_attention(q, k, v, None, BQ, BK, md)
    taken = _native.load().sa_fwd_split_workspace_bytes(B, H, Sq, Sk, D, BQ, BK, 0)
    assert taken > 0
    md = compute_mask_kernel(mask, BQ, BK, list_stats=True)
    torch.cuda.synchronize()
    torch.cuda.reset_peak_memory_stats()
    before = torch.cuda.memory_allocated()
    got = sparse_attention(q, k, v, None, BQ, BK, md)
    assert (torch.cuda.max_memory_allocated() - before < taken) == (keys == 512)  # (lists of eight chunks and of nine)
    assert torch.equal(got, want)
