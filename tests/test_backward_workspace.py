"""How much memory the backward takes for dS: never more than a quarter of what there is, and the same gradients from less."""
import math

import pytest
import torch

from sparseattention_amd import _native

GiB = 1 << 30
SIZES = [(8, 16, 4096, 4096), (1, 9, 16384, 16384), (2, 32, 1024, 1024), (1, 57, 128, 1152), (8, 32, 32768, 32768), (1, 8, 1024, 1024)]


@pytest.mark.parametrize("B,H,Sq,Sk", SIZES)
@pytest.mark.parametrize("D", [64, 128])
def test_bytes_within_a_limit(B, H, Sq, Sk, D):
    lib = _native.load()
    least, most = lib.sa_bwd_workspace_bytes(B, H, Sq), lib.sa_bwd_workspace_bytes_ex(B, H, Sq, Sk, D)
    before = 0
    for limit in sorted([0, 1, least, least + 2048, *(least + 1024 + (64 << 20 << i) for i in range(8)), most - 1, most, 1 << 50]):
        n = lib.sa_bwd_workspace_bytes_within(B, H, Sq, Sk, D, limit)
        assert max(least, before) <= n <= min(max(limit, least), most)
        # a workspace of that size has a use for all of it, for whole planes of at least 512 key tiles
        assert lib.sa_bwd_workspace_bytes_within(B, H, Sq, Sk, D, n) == n
        if n > least:
            planes = (n - least) // (Sq * Sk * 2)
            assert 0 <= n - least - planes * Sq * Sk * 2 < 1024 and planes * (Sk // 128) >= 512
        before = n
    assert lib.sa_bwd_workspace_bytes_within(B, H, Sq, Sk, D, most) == most


def test_a_quarter_of_the_room():
    host, lib = _native.host(), _native.load()
    args = (8, 16, 4096, 4096, 128)
    most, least = lib.sa_bwd_workspace_bytes_ex(*args), lib.sa_bwd_workspace_bytes(*args[:3])
    assert host.backward_workspace_bytes(*args, 200 * GiB) == most > 4 * GiB
    some = host.backward_workspace_bytes(*args, 8 * GiB)
    assert GiB < some <= 2 * GiB
    assert host.backward_workspace_bytes(*args, GiB) == host.backward_workspace_bytes(*args, 0) == least


@pytest.mark.gpu
def test_gradients_do_not_depend_on_the_planes_at_a_time(gpu):
    from sparseattention_amd import compute_backward_metadata, sparse_attention, workloads as W

    B, H, S, D = 2, 96, 1024, 128
    q, k, v = W.qkv(B, H, S, D, torch.bfloat16, seed=9, device=gpu)
    do = torch.randn_like(q)
    mask = torch.ones(S, S, dtype=torch.bool, device=gpu).tril()[None, None].expand(B, H, S, S)
    o, lse = sparse_attention(q, k, v, mask, 128, 64, return_lse=True)
    bmd = compute_backward_metadata(mask)
    lib, st = _native.load(), _native.strides
    lists, packs = [], []
    for md in (bmd.by_query, bmd.by_key):
        for t in (md.unmasked_kv_ids, md.unmasked_lens, md.masked_kv_ids, md.masked_lens):
            lists += [t.data_ptr(), st(t.stride())]
        packs += [md.packed_masks.data_ptr(), st(md.packed_masks.stride()[:2])]

    def gradients(nbytes):
        out = [torch.empty_like(t) for t in (q, k, v)]
        # (NaN patterns in whatever no pass writes)
        ws = torch.full((nbytes,), 0xFF, dtype=torch.uint8, device=gpu)
        tensors = [x for t in (q, k, v, o, do, lse, *out) for x in (t.data_ptr(), st(t.stride()))]
        _native.check(lib.sa_sparse_attention_bwd(*tensors, None, None, None, None, *packs, *lists, ws.data_ptr(), nbytes, B, H, S, S, D,
                                                  _native.SA_DTYPE_BF16, D ** -0.5 / math.log(2), torch.cuda.current_stream().cuda_stream))
        return out

    least, most = lib.sa_bwd_workspace_bytes(B, H, S), lib.sa_bwd_workspace_bytes_ex(B, H, S, S, D)
    want = gradients(most)
    for planes in (64, 100):
        nbytes = lib.sa_bwd_workspace_bytes_within(B, H, S, S, D, least + 1024 + planes * S * S * 2)
        assert least < nbytes < most
        assert all(torch.equal(a, b) for a, b in zip(gradients(nbytes), want))
    for a, b in zip(gradients(least), want):  # none stored: within rounding (both within 3.2e-3 of float64)
        assert float((a.double() - b.double()).norm() / b.double().norm()) <= 6.4e-3


@pytest.mark.gpu
def test_capture(gpu):
    """The look at the device's memory is no hindrance to a graph."""
    from sparseattention_amd import compute_backward_metadata, sparse_attention, sparse_attention_backward, workloads as W

    B, H, S, D = 1, 64, 1024, 128
    assert _native.load().sa_bwd_workspace_bytes_ex(B, H, S, S, D) > _native.load().sa_bwd_workspace_bytes(B, H, S)
    q, k, v = W.qkv(B, H, S, D, torch.bfloat16, seed=9, device=gpu)
    do = torch.randn_like(q)
    mask = torch.ones(S, S, dtype=torch.bool, device=gpu).tril()[None, None].expand(B, H, S, S)
    o, lse = sparse_attention(q, k, v, mask, 128, 64, return_lse=True)
    bmd = compute_backward_metadata(mask)
    sparse_attention_backward(do, q, k, v, o, lse, None, bmd)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        got = sparse_attention_backward(do, q, k, v, o, lse, None, bmd)
    for _ in range(3):
        do.copy_(torch.randn_like(do))
        graph.replay()
        want = sparse_attention_backward(do, q, k, v, o, lse, None, bmd)
        assert all(torch.equal(a, b) for a, b in zip(got, want))
