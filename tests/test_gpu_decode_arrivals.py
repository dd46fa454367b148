"""Decode whose last workgroup merges the parts (few of them, the larger workspace), against the merge by a second launch: the parts of a
row are added up in the same order, so the bits are the same, however large the workspace."""
import ctypes
import math

import pytest
import torch

from sparseattention_amd import _native, compute_mask_kernel, workloads as W

pytestmark = pytest.mark.gpu


def decode(q, k, v, md, BK, n, ws, ws_bytes, o, lse):
    S, (B, H, Sq, D), Sk = _native.strides, q.shape, k.shape[2]
    args = []
    for t in (q, k, v, o):
        args += [t.data_ptr(), S(t.stride())]
    args += [None, None]
    for t in (md.unmasked_kv_ids, md.unmasked_lens, md.masked_kv_ids, md.masked_lens):
        args += [t.data_ptr(), S(t.stride())]
    args += [md.packed_masks.data_ptr(), S(md.packed_masks.stride()[:2])]
    dt = _native.SA_DTYPE_BF16 if q.dtype == torch.bfloat16 else _native.SA_DTYPE_FP16
    rc = _native.load().sa_sparse_attention_decode_ex(
        *args, B, H, Sq, Sk, D, BK, dt, D ** -0.5 / math.log(2), n, ws.data_ptr(), ws_bytes, lse.data_ptr(), S(lse.stride()),
        ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    assert rc == 0, _native.load().sa_last_error()


# (parts of one row and of several; planes that start between two pieces of 16 bytes; the most rows there can be, of both head dims;
# then, one at a time, a part, a row or a partial row too many: the second launch merges whatever the workspace)
@pytest.mark.parametrize("D,Sq,n,merges", [(128, 1, 2, True), (128, 1, 3, True), (64, 1, 7, True), (64, 3, 5, True), (128, 16, 8, True),
                                           (64, 16, 2, True), (64, 4, 8, True), (128, 1, 9, False), (128, 1, 128, False), (128, 17, 2, False),
                                           (128, 32, 4, False), (64, 5, 7, False), (64, 32, 3, False), (64, 5, 25, False)])
def test_the_last_workgroup_merges(gpu, D, Sq, n, merges):
    B, H, Sk, BK = 3, 3, 8192, 64
    dtype = torch.bfloat16 if D == 128 else torch.float16
    q, k, v = W.qkv(B, H, Sq, D, dtype, seed=n, device=gpu, Sk=Sk)
    mask = torch.zeros(B, H, Sq, Sk, dtype=torch.bool, device=gpu)
    mask[0, :, :, :6000] = True
    mask[1, :, :, ::97] = True
    mask[2, 0, :, 64:70] = True  # (all parts but one are empty; the other heads' planes have none)
    md = compute_mask_kernel(mask, Sq, BK)
    lib = _native.load()
    least, more = lib.sa_decode_workspace_bytes(B, H, Sq, D, n), lib.sa_decode_workspace_bytes_ex(B, H, Sq, D, n)
    assert more == (least + 8 * B * H if merges else least)
    more = least + 8 * B * H  # (what a caller with one workspace for all calls has)
    out = lambda: (torch.empty_like(q), torch.empty(B, H, Sq, device=gpu))  # noqa: E731
    ws = torch.empty(more + 64, dtype=torch.uint8, device=gpu)
    want = out()
    decode(q, k, v, md, BK, n, ws, least, *want)
    torch.cuda.synchronize()
    for fill in (0, 255, 127, None):  # whatever the memory held; last, what a call left
        if fill is not None:
            ws.fill_(fill)
        got = out()
        decode(q, k, v, md, BK, n, ws, more, *got)
        torch.cuda.synchronize()
        if fill is not None:
            assert (ws[more:] == fill).all()
        assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])


def test_replays_bring_the_same_launch_number(gpu):
    B, H, Sq, Sk, D, BK, n = 2, 3, 2, 4096, 128, 64, 6
    q, k, v = W.qkv(B, H, Sq, D, torch.bfloat16, seed=5, device=gpu, Sk=Sk)
    mask = torch.rand(1, 1, Sq, Sk, device=gpu, generator=torch.Generator(gpu).manual_seed(1)) < 0.6
    md = compute_mask_kernel(mask.expand(B, H, Sq, Sk), Sq, BK)
    more = _native.load().sa_decode_workspace_bytes_ex(B, H, Sq, D, n)
    ws = torch.zeros(more, dtype=torch.uint8, device=gpu)
    o, lse = torch.empty_like(q), torch.empty(B, H, Sq, device=gpu)
    decode(q, k, v, md, BK, n, ws, more, o, lse)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        decode(q, k, v, md, BK, n, ws, more, o, lse)
    for i in range(4):
        q.copy_(torch.randn_like(q))
        want, wlse = torch.empty_like(q), torch.empty_like(lse)
        if i == 2:
            ws.fill_(37)
        graph.replay()
        torch.cuda.synchronize()
        got, glse = o.clone(), lse.clone()
        decode(q, k, v, md, BK, n, torch.empty_like(ws), more, want, wlse)
        torch.cuda.synchronize()
        assert torch.equal(got, want) and torch.equal(glse, wlse)
