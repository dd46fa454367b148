"""Lists with assistants (up to one Q tile of 128 rows a compute unit): a second workgroup takes the end of a list that is longer than that
of the tile it shares a compute unit with, and the last of the two to finish adds the parts up."""
import ctypes
import gc
import math

import pytest
import torch

from sparseattention_amd import MaskMetadata, _native, compute_mask_kernel, sparse_attention, workloads as W
from sparseattention_amd.mask_utils import validation_key

pytestmark = pytest.mark.gpu


def _masks(S, B, gpu):
    i = torch.arange(S, device=gpu)
    causal = i[None] <= i[:, None]
    uneven = causal.clone()
    uneven[128:256] = True        # the longest lists where short ones are expected
    uneven[S - 128:] = False      # and a tile without any
    uneven[5, :] = False
    return {"causal": causal[None].expand(B, S, S), "every key": torch.ones(B, S, S, dtype=torch.bool, device=gpu),
            "uneven": uneven[None].expand(B, S, S),
            "blocks": torch.stack([W.random_block_mask(S, 64, 0.5, seed=b, device=gpu) for b in range(B)])}


# (planes x Q tiles: 256, fewer tiles than compute units, one and three planes to an XCD; lists of whole and of half chunks, of several)
@pytest.mark.parametrize("B,H,S,D,BK,dtype", [(1, 32, 1024, 128, 64, torch.bfloat16), (1, 16, 2048, 128, 32, torch.bfloat16),
                                              (3, 8, 1152, 128, 128, torch.float16), (1, 8, 2304, 128, 256, torch.bfloat16),
                                              (1, 16, 1664, 64, 32, torch.float16), (1, 8, 3072, 64, 64, torch.bfloat16),
                                              (1, 24, 1280, 128, 64, torch.float16)])
@pytest.mark.parametrize("case", ["causal", "every key", "uneven", "blocks"])
def test_outputs_and_lse(gpu, B, H, S, D, BK, dtype, case):
    assert 128 < B * H * S // 128 <= 256
    q, k, v = W.qkv(B, H, S, D, dtype, seed=S + BK, device=gpu)
    mask = _masks(S, B, gpu)[case][:, None].expand(B, H, S, S)
    md = compute_mask_kernel(mask, 128, BK)
    assert _native.host().forward_lists(q, S, 128, BK, md) == "shared"
    for m in (md, compute_mask_kernel(mask, 128, BK, pack_partial=False)):
        o, lse = sparse_attention(q, k, v, mask, 128, BK, mask_metadata=m, return_lse=True)
        s = (q.float() @ k.float().transpose(-1, -2).contiguous()) * D ** -0.5
        s = s.masked_fill(~mask, float("-inf"))
        want = (torch.softmax(s, -1).nan_to_num() @ v.float())
        assert float((o.float() - want).abs().max()) <= (2e-2 if dtype == torch.bfloat16 else 4e-3)
        want_lse = torch.logsumexp(s, -1)
        assert torch.equal(lse == float("-inf"), want_lse == float("-inf"))
        live = want_lse != float("-inf")
        assert float((lse[live] - want_lse[live]).abs().max()) <= 6e-3
        again = sparse_attention(q, k, v, mask, 128, BK, mask_metadata=m)
        assert torch.equal(o, again)  # whoever adds up: in the order of the parts


def test_replays_of_a_captured_launch(gpu):
    B, H, S = 1, 32, 1024
    q, k, v = W.qkv(B, H, S, 128, torch.bfloat16, seed=9, device=gpu)
    mask = _masks(S, B, gpu)["causal"][:, None].expand(B, H, S, S)
    md = compute_mask_kernel(mask, 128, 64)
    want = sparse_attention(q, k, v, mask, 128, 64, mask_metadata=md)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        o = sparse_attention(q, k, v, mask, 128, 64, mask_metadata=md)
    for _ in range(4):
        o.fill_(7.0)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(o, want)
        assert torch.equal(sparse_attention(q, k, v, mask, 128, 64, mask_metadata=md), want)


def test_a_workspace_without_room_goes_without_assistants(gpu):
    """None, one that is too small, one whose address does not suit: the plain form, as for callers of a library that asked for none."""
    B, H, S = 1, 32, 1024
    q, k, v = W.qkv(B, H, S, 128, torch.bfloat16, seed=4, device=gpu)
    mask = _masks(S, B, gpu)["causal"][:, None].expand(B, H, S, S)
    md = compute_mask_kernel(mask, 128, 64)
    lib, st = _native.load(), lambda t: _native.strides(t.stride())
    need = lib.sa_fwd_split_workspace_bytes(B, H, S, S, 128, 128, 64, 0)
    assert need >= 2 * 256 * 128 * 130 * 4 + 16 * 256

    def call(ws, nbytes):
        o = torch.empty_like(q)
        pk = (md.packed_masks.data_ptr(), _native.strides(md.packed_masks.stride()[:2]))
        rc = lib.sa_sparse_attention_fwd_split(
            q.data_ptr(), st(q), k.data_ptr(), st(k), v.data_ptr(), st(v), o.data_ptr(), st(o), None, None, md.unmasked_kv_ids.data_ptr(),
            st(md.unmasked_kv_ids), md.unmasked_lens.data_ptr(), st(md.unmasked_lens), md.masked_kv_ids.data_ptr(), st(md.masked_kv_ids),
            md.masked_lens.data_ptr(), st(md.masked_lens), *pk, None, None, B, H, S, S, 128, 128, 64, 0, 128 ** -0.5 / math.log(2), ws, nbytes,
            ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
        assert rc == 0, lib.sa_last_error()
        return o

    ws = torch.empty(need + 32, dtype=torch.uint8, device=gpu)
    plain = call(None, 0)
    assert torch.equal(call(ws.data_ptr(), 64), plain) and torch.equal(call(ws.data_ptr(), need - 8), plain)
    assert torch.equal(call(ws.data_ptr() + 8, need), plain)
    o = call(ws.data_ptr(), need)
    assert torch.equal(o, sparse_attention(q, k, v, mask, 128, 64, mask_metadata=md)) and not torch.equal(o, plain)
    assert float((o.float() - plain.float()).abs().max()) <= 2e-2


@pytest.mark.parametrize("BK", [32, 64, 128])
def test_lists_known_to_be_alike_have_no_assistants(gpu, BK):
    """Statistics that say by how much the longest list exceeds the mean: less than six chunks of 64 keys stay with one workgroup each."""
    B, H, S = 1, 16, 2048
    q, k, v = W.qkv(B, H, S, 128, torch.bfloat16, seed=5, device=gpu)
    assert _native.load().sa_fwd_split_uneven_keys(B, H, S, S, 128, 128, BK, 0) == 6 * 64
    tile = torch.arange(S, device=gpu) // 128
    for longer in (0, 3, 4, 8):  # blocks of 128 keys that one of the 16 Q tiles has beyond the others' eight: 15/16 of them is what it exceeds the mean by
        mask = ((tile[None] < 8) | ((tile[:, None] == 15) & (tile[None] < 8 + longer)))[None, None].expand(B, H, S, S)
        known, unknown = compute_mask_kernel(mask, 128, BK, list_stats=True), compute_mask_kernel(mask, 128, BK)
        assert (known.list_stats[1] - known.list_stats[0]) * BK == longer * 120
        assert _native.host().forward_lists(q, S, 128, BK, unknown) == "shared"
        assert _native.host().forward_lists(q, S, 128, BK, known) == ("whole" if longer * 120 < 384 else "shared")
        o = sparse_attention(q, k, v, mask, 128, BK, mask_metadata=known, kernel="default")
        want = torch.softmax((q.float() @ k.float().transpose(-1, -2).contiguous() * 128 ** -0.5).masked_fill(~mask, float("-inf")), -1) @ v.float()
        assert float((o.float() - want).abs().max()) <= 2e-2


def _without_room(fn):
    """fn() with 16 MiB in one piece for it to allocate, and less than 2 MiB anywhere else."""
    gc.collect()
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    room, filled = torch.empty(16 << 20, dtype=torch.uint8, device="cuda"), []
    torch.cuda.set_per_process_memory_fraction(torch.cuda.memory_reserved() / torch.cuda.get_device_properties(0).total_memory)
    try:
        for size in (64 << 20, 8 << 20, 2 << 20):  # (what other tensors left free of their segments)
            try:
                while True:
                    filled.append(torch.empty(size, dtype=torch.uint8, device="cuda"))
            except torch.OutOfMemoryError:
                pass
        del room
        return fn()
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)


def test_no_memory_for_parts(gpu):
    """Assistants are done without where their parts find no place, as such launches asked for none once.  A launch whose lists are shared
    for their length says that it has no memory."""
    B, H, S = 1, 32, 1024
    q, k, v = W.qkv(B, H, S, 128, torch.bfloat16, seed=6, device=gpu)
    mask = _masks(S, B, gpu)["causal"][:, None].expand(B, H, S, S)
    md = compute_mask_kernel(mask, 128, 64)
    assert _native.load().sa_fwd_split_workspace_bytes(B, H, S, S, 128, 128, 64, 0) > 32 << 20
    with_parts = sparse_attention(q, k, v, mask, 128, 64, mask_metadata=md)
    got = _without_room(lambda: sparse_attention(q, k, v, mask, 128, 64, mask_metadata=md))
    even = compute_mask_kernel(mask, 128, 64)
    even.list_stats = (16.0, 16)  # (statistics that keep the lists whole)
    assert torch.equal(got, sparse_attention(q, k, v, mask, 128, 64, mask_metadata=even, kernel="default"))
    assert not torch.equal(got, with_parts) and float((got.float() - with_parts.float()).abs().max()) <= 2e-2

    q, k, v = (torch.randn(1, 32, s, 128, device=gpu, dtype=torch.bfloat16) for s in (512, 8192, 8192))
    mask = torch.ones(1, 1, 512, 8192, dtype=torch.bool, device=gpu).expand(1, 32, 512, 8192)
    md = compute_mask_kernel(mask, 128, 64)
    lib = _native.load()
    assert lib.sa_fwd_split_workspace_bytes(1, 32, 512, 8192, 128, 128, 64, 0) > 24 << 20 and lib.sa_fwd_split_uneven_keys(1, 32, 512, 8192, 128, 128, 64, 0) == 0
    want = sparse_attention(q, k, v, mask, 128, 64, mask_metadata=md)
    with pytest.raises(torch.OutOfMemoryError):
        _without_room(lambda: sparse_attention(q, k, v, mask, 128, 64, mask_metadata=md))
    assert torch.equal(sparse_attention(q, k, v, mask, 128, 64, mask_metadata=md), want)


def test_projections_seen_through_a_transpose(gpu):
    B, H, S = 3, 8, 1152
    q, k, v = (torch.randn(B, S, H, 128, device=gpu, generator=torch.Generator(device=gpu).manual_seed(i)).to(torch.bfloat16).transpose(1, 2) for i in range(3))
    mask = _masks(S, B, gpu)["causal"][:, None].expand(B, H, S, S)
    md = compute_mask_kernel(mask, 128, 64)
    assert _native.host().forward_lists(q, S, 128, 64, md) == "shared"
    o, lse = sparse_attention(q, k, v, mask, 128, 64, mask_metadata=md, return_lse=True)
    o2, lse2 = sparse_attention(q.contiguous(), k.contiguous(), v.contiguous(), mask, 128, 64, mask_metadata=md, return_lse=True)
    assert torch.equal(o, o2) and torch.equal(lse, lse2)


@pytest.mark.parametrize("D", [64, 128])
def test_infinite_values_that_lists_name(gpu, D):
    """An infinity or a NaN in V reaches its column of the result whichever part names it, and no other column."""
    B, H, S = 1, 16, 2048
    q, k, v = W.qkv(B, H, S, D, torch.bfloat16, seed=5, device=gpu)
    mask = _masks(S, 1, gpu)["causal"][:, None].expand(B, H, S, S)
    want = torch.softmax((q.double() @ k.double().transpose(-1, -2).contiguous() * D ** -0.5).masked_fill(~mask, float("-inf")), -1) @ v.double()
    # (the last tiles have an assistant: the first of these keys are in the first part of their lists, the second ones in the end of it)
    v[..., 70, 3], v[..., 1800, 9] = float("inf"), float("-inf")
    v[..., 90, 17], v[..., 1810, 31] = float("nan"), float("nan")
    md = compute_mask_kernel(mask, 128, 64)
    assert _native.host().forward_lists(q, S, 128, 64, md) == "shared"
    o = sparse_attention(q, k, v, mask, 128, 64, mask_metadata=md).double()
    far, near = slice(1920, S), slice(128, 1664)  # (of a tile that names a key every row has it, by a weight of 0 where it does not attend)
    assert torch.isposinf(o[:, :, far, 3]).all() and torch.isneginf(o[:, :, far, 9]).all()
    assert torch.isnan(o[:, :, far, 17]).all() and torch.isnan(o[:, :, far, 31]).all()
    assert torch.isposinf(o[:, :, near, 3]).all() and torch.isnan(o[:, :, near, 17]).all()
    assert torch.isfinite(o[:, :, near, 9]).all() and torch.isfinite(o[:, :, near, 31]).all()
    rest = [d for d in range(D) if d not in (3, 9, 17, 31)]
    assert float((o[..., rest] - want[..., rest]).norm() / want[..., rest].norm()) <= 2.0 ** -7


def test_entries_out_of_range(gpu):
    """An entry outside K leaves other Q tiles alone and is left out, in the first part of a list and in the assistant's."""
    B, H, S, BK = 1, 16, 2048, 64
    q, k, v = W.qkv(B, H, S, 128, torch.bfloat16, seed=7, device=gpu)
    tile = torch.arange(S, device=gpu) // 128
    mask = (tile[None] <= tile[:, None])[None, None].expand(B, H, S, S)  # FULL tiles only, two a block of 128 keys
    md = compute_mask_kernel(mask, 128, BK)
    o = sparse_attention(q, k, v, mask, 128, BK, mask_metadata=md)
    ids = md.unmasked_kv_ids.clone()
    ids[..., 15, 3], ids[..., 15, 29] = S // BK, -1  # of the longest list: 32 entries, of which the assistant takes 15
    bad = MaskMetadata(ids, md.unmasked_lens.clone(), md.masked_kv_ids, md.masked_lens, md.packed_masks)
    bad._validated_for = validation_key(bad, S, BK)  # (past the wrapper's own check)
    assert _native.host().forward_lists(q, S, 128, BK, bad) == "shared"
    got = sparse_attention(q, k, v, mask, 128, BK, mask_metadata=bad)
    assert torch.equal(got[:, :, :1920], o[:, :, :1920])
    left = mask[:, :, 1920:].clone()
    for e in (3, 29):
        left[..., BK * e:BK * (e + 1)] = False
    want = torch.softmax((q[:, :, 1920:].double() @ k.double().transpose(-1, -2).contiguous() * 128 ** -0.5).masked_fill(~left, float("-inf")), -1) @ v.double()
    assert float((got[:, :, 1920:].double() - want).norm() / want.norm()) <= 2.0 ** -7


def test_no_further_from_float64_than_one_workgroup_a_list(gpu):
    """Two reference values instead of one: 46 cases of other sizes, masks and seeds were all nearer by 0.003 to 0.07 %; ten times the least of it."""
    B, H, S = 1, 32, 1024
    q, k, v = W.qkv(B, H, S, 128, torch.bfloat16, seed=11, device=gpu)
    mask = _masks(S, B, gpu)["causal"][:, None].expand(B, H, S, S)
    want = torch.softmax((q.double() @ k.double().transpose(-1, -2).contiguous() * 128 ** -0.5).masked_fill(~mask, float("-inf")), -1) @ v.double()
    md, whole = compute_mask_kernel(mask, 128, 64), compute_mask_kernel(mask, 128, 64)
    whole.list_stats = (16.0, 16)  # (statistics that keep the lists whole)
    off = [float((sparse_attention(q, k, v, mask, 128, 64, mask_metadata=m, kernel="default").double() - want).norm() / want.norm()) for m in (md, whole)]
    assert off[0] != off[1] and off[0] <= off[1] * 1.0003
