"""Which launches walk their lists in two halves: the edges of the rule, and metadata that says that all lists are short."""
import pytest
import torch

from sparseattention_amd import _native, compute_mask_kernel, sparse_attention, workloads as W

pytestmark = pytest.mark.gpu


def handed_out(gpu, tiles, Sk, D, BQ, BK, md=None, dtype=torch.bfloat16):
    q = torch.empty(1, tiles, BQ, D, dtype=dtype, device=gpu)
    return _native.host().forward_lists(q, Sk, BQ, BK, md)


# (chunks of 64 keys up to which one workgroup of half the waves is no slower)
@pytest.mark.parametrize("D,BQ,least", [(128, 128, 16), (64, 128, 13), (128, 64, 5), (64, 64, 5)])
@pytest.mark.parametrize("packed", [True, False])
def test_lists_known_to_be_short_stay_whole(gpu, D, BQ, least, packed):
    cus = torch.cuda.get_device_properties(gpu).multi_processor_count
    H, Sk, BK = 4, 4096, 64
    Sq = BQ * (cus // H)
    q, _, _ = W.qkv(1, H, Sq, D, torch.bfloat16, seed=1, device=gpu)
    _, k, v = W.qkv(1, H, Sk, D, torch.bfloat16, seed=2, device=gpu)
    assert _native.load().sa_fwd_split_workspace_bytes(1, H, Sq, Sk, D, BQ, BK, 0) == 0
    assert _native.load().sa_fwd_split_least_keys(1, H, Sq, Sk, D, BQ, BK, 0) == 64 * least
    for chunks in (1, least, least + 1):
        mask = torch.zeros(1, 1, Sq, Sk, dtype=torch.bool, device=gpu)
        mask[..., 3:64 * chunks] = True
        mask[..., : Sq // 2, 64:] = False
        me = mask.expand(1, H, Sq, Sk)
        known = compute_mask_kernel(me, BQ, BK, pack_partial=packed, list_stats=True)
        unknown = compute_mask_kernel(me, BQ, BK, pack_partial=packed)
        assert known.list_stats[1] == chunks
        assert handed_out(gpu, cus, Sk, D, BQ, BK, known) == ("whole" if chunks <= least else "halves")
        assert handed_out(gpu, cus, Sk, D, BQ, BK, unknown) == "halves"
        o, lse = sparse_attention(q, k, v, me, BQ, BK, mask_metadata=known, return_lse=True, kernel="default")
        other, other_lse = sparse_attention(q, k, v, me, BQ, BK, mask_metadata=unknown, return_lse=True, kernel="default")
        s = (q[0].double() @ k[0].double().transpose(-1, -2).contiguous()) * D ** -0.5
        s = s.masked_fill(~mask[0], float("-inf"))
        want = torch.softmax(s, -1) @ v[0].double()
        # P and the output are rounded to 8 bits: half a unit of each, and as much of the scaled queries
        for got, got_lse in ((o, lse), (other, other_lse)):
            assert float((got[0].double() - want).norm() / want.norm()) <= 2 * 2.0 ** -8
            assert float((got_lse[0] - torch.logsumexp(s, -1)).abs().max()) <= 16 * 2.0 ** -8


def test_edges_of_the_rule(gpu):
    cus = torch.cuda.get_device_properties(gpu).multi_processor_count
    if cus % 4:
        pytest.skip("the edges lie at parts of the compute units")
    halves = [  # tiles, chunks, D, BLOCK_Q, BLOCK_K
        (cus, 96, 128, 128, 64), (cus, 49, 64, 128, 32), (cus - 1, 72, 128, 128, 64), (cus // 2 + 1, 49, 128, 128, 1024),
        (cus // 2 + 1, 16, 128, 64, 64), (cus, 16, 64, 64, 32), (cus // 2 + 1, 96, 64, 64, 64), (cus, 256, 128, 64, 64),
        (3 * cus // 4, 256, 128, 64, 64), (cus - 1, 256, 64, 64, 64)]
    other = [
        (cus, 97, 128, 128, 64), (cus, 48, 128, 128, 64), (cus - 1, 73, 128, 128, 64), (cus // 2, 49, 128, 128, 64), (cus + 1, 64, 128, 128, 64),
        (cus, 64, 128, 128, 16), (cus // 2, 16, 128, 64, 64), (cus, 15, 64, 64, 64), (cus + 1, 16, 64, 64, 64), (cus, 16, 64, 64, 16),
        (2 * cus // 3, 97, 64, 64, 64), (3 * cus // 4 + 1, 97, 128, 64, 64), (cus, 64, 128, 32, 64), (cus, 64, 256, 128, 64)]
    for tiles, chunks, D, BQ, BK in halves:
        Sk = -(-64 * chunks // BK) * BK
        assert handed_out(gpu, tiles, Sk, D, BQ, BK) == "halves", (tiles, chunks, D, BQ, BK)
        assert handed_out(gpu, tiles, Sk, D, BQ, BK, dtype=torch.float32) != "halves", (tiles, chunks, D, BQ, BK)
    for tiles, chunks, D, BQ, BK in other:
        assert handed_out(gpu, tiles, 64 * chunks, D, BQ, BK) != "halves", (tiles, chunks, D, BQ, BK)
