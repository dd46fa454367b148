"""Shared lists whose last workgroup adds the parts up (the whole workspace) against the merge by a second launch (a workspace without
place for the workgroups' words) and against the definition."""
import ctypes
import dataclasses
import math

import pytest
import torch

from sparseattention_amd import _native, compute_mask_kernel, workloads as W

pytestmark = pytest.mark.gpu

CODE = {torch.bfloat16: 0, torch.float16: 1, torch.float32: 2}
# a result's own rounding (2^-9, 2^-12 of values up to 4) with that of P, twice; float32: a row's sum of 4096 terms in another order
TOL = {torch.bfloat16: 2e-2, torch.float16: 4e-3, torch.float32: 1e-5}


def forward(q, k, v, md, BQ, BK, ws, ws_bytes, o, lse):
    S, (B, H, Sq, D), Sk = _native.strides, q.shape, k.shape[2]
    args = []
    for t in (q, k, v, o):
        args += [t.data_ptr(), S(t.stride())]
    args += [None, None]
    for t in (md.unmasked_kv_ids, md.unmasked_lens, md.masked_kv_ids, md.masked_lens):
        args += [t.data_ptr(), S(t.stride())]
    args += [md.packed_masks.data_ptr(), S(md.packed_masks.stride()[:2]), lse.data_ptr(), S(lse.stride())]
    rc = _native.load().sa_sparse_attention_fwd_split(*args, B, H, Sq, Sk, D, BQ, BK, CODE[q.dtype], D ** -0.5 / math.log(2), ws.data_ptr(),
                                                      ws_bytes, ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    assert rc == 0, _native.load().sa_last_error()


def sizes_of(q, Sk, BQ, BK):
    """(bytes with the words, where the launch has them; bytes of the parts alone)"""
    B, H, Sq, D = q.shape
    full = _native.load().sa_fwd_split_workspace_bytes(B, H, Sq, Sk, D, BQ, BK, CODE[q.dtype])
    tiles, part = B * H * (Sq // BQ), BQ * (D + 2) * 4
    return full, full if full % (tiles * (part + 8)) else full // (part + 8) * part


def sizes(q, Sk, BQ, BK):
    """(bytes with the words, bytes of the parts alone)"""
    full, parts = sizes_of(q, Sk, BQ, BK)
    assert 0 < parts < full
    return full, parts


def uneven(B, H, Sq, Sk, BQ, gpu):
    """Lists from none to all tiles, FULL, PARTIAL and EMPTY ones in turn; rows that attend to nothing."""
    mask = torch.rand(B, 1, Sq, Sk, generator=torch.Generator().manual_seed(Sk)) < 0.5
    for c in range(0, Sk, 256):
        mask[..., c:c + 64] = True
        mask[..., c + 64:c + 128] = False
    mask[:, :, 3] = False
    mask[0, 0, :BQ, Sk // 2 + 5:] = False  # (parts without a key)
    mask[-1, 0, Sq - BQ:, 33:] = False     # one short list
    mask[-1, 0, Sq - BQ:, :33] = True
    return mask.to(gpu).expand(B, H, Sq, Sk)


@pytest.mark.parametrize("dtype,B,H,Sq,Sk,D,BQ,BK", [
    (torch.float32, 1, 4, 512, 512, 64, 64, 32),      # two groups of waves
    (torch.float32, 1, 3, 192, 160, 64, 64, 16),      # an odd number of chunks: one group has one more
    (torch.float32, 1, 2, 64, 1280, 64, 32, 16),      # lists that come by way of LDS; one wave a group
    (torch.float32, 1, 2, 128, 1024, 64, 64, 256),    # entries of several chunks, shared out between the groups
    (torch.float32, 1, 2, 128, 256, 128, 64, 32),
    (torch.float32, 2, 16, 512, 160, 128, 128, 32),   # one group of four waves
    (torch.bfloat16, 4, 8, 512, 4096, 128, 128, 64),  # four parts of four waves
    (torch.bfloat16, 1, 9, 256, 2048, 128, 128, 32),
    (torch.float16, 3, 8, 256, 2560, 64, 64, 16),     # parts that do not divide the list
    (torch.float16, 1, 2, 96, 2048, 64, 32, 64),      # one wave
    (torch.bfloat16, 1, 2, 64, 2048, 128, 64, 1024),  # entries of several chunks, fewer than parts
])
def test_the_last_workgroup_adds_up(gpu, dtype, B, H, Sq, Sk, D, BQ, BK):
    q, _, _ = W.qkv(B, H, Sq, D, dtype, seed=1, device=gpu)
    _, k, v = W.qkv(B, H, Sk, D, dtype, seed=2, device=gpu)
    mask = uneven(B, H, Sq, Sk, BQ, gpu)
    md = compute_mask_kernel(mask, BQ, BK)
    full, parts = sizes(q, Sk, BQ, BK)
    out = lambda: (torch.empty_like(q), torch.empty(B, H, Sq, device=gpu))  # noqa: E731
    ws = torch.empty(full + 64, dtype=torch.uint8, device=gpu)
    two, one = out(), out()
    forward(q, k, v, md, BQ, BK, ws, parts, *two)
    for fill in (255, 0, None):  # whatever the memory held; last, what a call left
        if fill is not None:
            ws.fill_(fill)
        got = out()
        forward(q, k, v, md, BQ, BK, ws, full, *got)
        torch.cuda.synchronize()
        if fill == 255:
            one = got
        assert torch.equal(got[0], one[0]) and torch.equal(got[1], one[1])  # (the parts in their order, whoever adds)
    s = ((q.double() @ k.double().transpose(-1, -2).contiguous()) * D ** -0.5).masked_fill(~mask, float("-inf"))
    want, want_lse = torch.nan_to_num(torch.softmax(s, -1)) @ v.double(), torch.logsumexp(s, -1)
    live = torch.isfinite(want_lse)
    for o, lse in (one, two):
        assert float((o.double() - want).abs().max()) <= TOL[dtype]
        assert torch.equal(torch.isfinite(lse), live)
        assert float((lse.double() - want_lse)[live].abs().max()) <= (1e-5 if dtype == torch.float32 else 6e-3 + 2 ** -9 * 5)


@pytest.mark.parametrize("dtype,B,H,Sq,Sk,D,BQ,BK", [(torch.float32, 1, 4, 256, 512, 64, 64, 32), (torch.bfloat16, 1, 9, 256, 2048, 128, 128, 64)])
def test_replays_bring_the_same_launch_number(gpu, dtype, B, H, Sq, Sk, D, BQ, BK):
    q, _, _ = W.qkv(B, H, Sq, D, dtype, seed=1, device=gpu)
    _, k, v = W.qkv(B, H, Sk, D, dtype, seed=2, device=gpu)
    md = compute_mask_kernel(uneven(B, H, Sq, Sk, BQ, gpu), BQ, BK)
    full, _ = sizes(q, Sk, BQ, BK)
    ws = torch.zeros(full, dtype=torch.uint8, device=gpu)
    o, lse = torch.empty_like(q), torch.empty(B, H, Sq, device=gpu)
    forward(q, k, v, md, BQ, BK, ws, full, o, lse)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        forward(q, k, v, md, BQ, BK, ws, full, o, lse)
    for i in range(4):
        q.copy_(torch.randn_like(q))
        want, wlse = torch.empty_like(q), torch.empty_like(lse)
        if i == 2:
            ws.fill_(37)
        graph.replay()
        torch.cuda.synchronize()
        got, glse = o.clone(), lse.clone()
        forward(q, k, v, md, BQ, BK, torch.empty_like(ws), full, want, wlse)
        torch.cuda.synchronize()
        assert torch.equal(got, want) and torch.equal(glse, wlse)


@pytest.mark.parametrize("B,H,Sq,Sk,D,BQ,BK", [
    (1, 4, 512, 512, 64, 64, 32),     # two groups of waves, 16 slots a row
    (1, 2, 64, 1280, 64, 32, 16),     # 80 slots: lists of more entries than lanes
    (1, 2, 128, 1024, 64, 64, 256),   # entries of several chunks
    (1, 4, 256, 160, 128, 128, 32),   # one group
])
def test_rows_that_end_with_the_longest_list(gpu, B, H, Sq, Sk, D, BQ, BK):
    """float32 reads ids[..., :len] alone: lists in rows of as many slots as the longest has, the last one at the end of its memory."""
    q, _, _ = W.qkv(B, H, Sq, D, torch.float32, seed=1, device=gpu)
    _, k, v = W.qkv(B, H, Sk, D, torch.float32, seed=2, device=gpu)
    md = compute_mask_kernel(uneven(B, H, Sq, Sk, BQ, gpu), BQ, BK)
    full, _ = sizes(q, Sk, BQ, BK)
    ws = torch.empty(full, dtype=torch.uint8, device=gpu)
    want, got = ((torch.empty_like(q), torch.empty(B, H, Sq, device=gpu)) for _ in range(2))
    forward(q, k, v, md, BQ, BK, ws, full, *want)
    ids = [(md.unmasked_kv_ids, md.unmasked_lens), (md.masked_kv_ids, md.masked_lens)]
    cut = [t[..., :max(1, int(n.max()))].contiguous() for t, n in ids]
    forward(q, k, v, dataclasses.replace(md, unmasked_kv_ids=cut[0], masked_kv_ids=cut[1]), BQ, BK, ws, full, *got)
    torch.cuda.synchronize()
    assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])


@pytest.mark.parametrize("tiles", [8, 16, 32, 48, 64, 80, 128])
def test_no_more_parts_than_run_at_once(gpu, tiles):
    """float32, D = 128, BLOCK_Q 64: a workgroup takes the LDS of its compute unit, so the launch has one for each; elsewhere two."""
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    D, Sk = 128, 4096
    for BQ, most in ((64, cus), (128, 2 * cus)):
        q = torch.empty(1, 1, tiles * BQ, D, dtype=torch.float32, device=gpu)
        _, parts = sizes_of(q, Sk, BQ, 32)
        assert parts // (tiles * BQ * (D + 2) * 4) == min(64, 32, most // tiles)


@pytest.mark.parametrize("dtype,tiles,BQ,Sk,in_launch", [
    (torch.bfloat16, 8, 128, 2048, False), (torch.bfloat16, 16, 128, 2048, False), (torch.bfloat16, 17, 128, 2048, True),
    (torch.bfloat16, 8, 64, 2048, True), (torch.bfloat16, 8, 64, 4096, False), (torch.float32, 8, 128, 256, True), (torch.float32, 8, 128, 512, False)])
def test_which_launch_adds_up(gpu, dtype, tiles, BQ, Sk, in_launch):
    """One workgroup adds up 256 KiB of 16-bit types' parts only where enough of them do so side by side."""
    q = torch.empty(1, 1, tiles * BQ, 128, dtype=dtype, device=gpu)
    full, parts = sizes_of(q, Sk, BQ, 64)
    assert (full > parts) == in_launch
