"""Lists with assistants (up to one Q tile of 128 rows a compute unit): a second workgroup takes the end of a list that is longer than that
of the tile it shares a compute unit with, and the last of the two to finish adds the parts up."""
import pytest
import torch

from sparseattention_amd import _native, compute_mask_kernel, sparse_attention, workloads as W

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
