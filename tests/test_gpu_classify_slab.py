"""Classification, lists and packed tiles of slabs of megabytes in one launch: rows whose last 16-byte pieces fill a column block or
part of one, with and without a second block to a wave, Q tiles that are no multiple of the rows in flight, planes of their own and
shared ones, rows apart in memory, and both sides of the rule's edges."""
import pytest
import torch

from sparseattention_amd import _native, compute_mask_kernel

pytestmark = pytest.mark.gpu

# (distinct batches, distinct heads, nQ, BQ, Sk, BK, columns between rows)
CASES = [(1, 1, 128, 128, 8192, 64, 8192), (1, 2, 96, 131, 8208, 16, 8208), (2, 1, 96, 128, 8192 + 96, 32, 8192 + 96),
         (1, 1, 192, 130, 16384 + 16, 16, 16384 + 512), (1, 1, 256, 128, 32768 - 128, 128, 32768), (1, 1, 256, 128, 32768 + 1024, 1024, 32768 + 1024),
         (1, 1, 256, 67, 32768 + 32, 32, 32768 + 32), (1, 1, 128, 67, 8192 + 1024, 1024, 8192 + 1024),
         (1, 1, 127, 128, 8192, 64, 8192), (1, 1, 192, 128, 8176, 16, 8176), (1, 1, 128, 64, 8192, 64, 8192),   # the three-launch and the small form
         (1, 1, 256, 67, 32768 + 16, 16, 32768 + 16)]                                                          # more tiles than LDS holds


@pytest.mark.parametrize("uB,uH,nQ,BQ,Sk,BK,pitch", CASES)
def test_lists_and_bits(gpu, uB, uH, nQ, BQ, Sk, BK, pitch):
    g = torch.Generator(device=gpu).manual_seed(BQ * Sk + BK)
    nK, Sq = Sk // BK, nQ * BQ
    u = torch.rand(uB, uH, nQ, 1, nK, 1, generator=g, device=gpu)
    dense = torch.rand(uB, uH, nQ, BQ, nK, BK, generator=g, device=gpu) < 0.5
    tiles = torch.where(u < 0.3, dense, u < 0.6)
    for only, value in ((0.6, True), (0.8, False)):                       # FULL but for one entry, empty but for one
        one = (u > only) & (u < only + 0.1)
        where = torch.randint(BQ * BK, (uB, uH, nQ, 1, nK, 1), generator=g, device=gpu)
        at = torch.arange(BQ, device=gpu).view(BQ, 1, 1) * BK + torch.arange(BK, device=gpu) == where
        tiles = torch.where(one, at != value, tiles)
    del dense
    store = torch.zeros(uB, uH, Sq, pitch, dtype=torch.bool, device=gpu)
    store[..., :Sk] = tiles.reshape(uB, uH, Sq, Sk)
    got = compute_mask_kernel(store[..., :Sk].expand(2, 2, Sq, Sk), BQ, BK)
    some, every = tiles.any(5).any(3), tiles.all(5).all(3)
    ids = torch.arange(nK, device=gpu, dtype=torch.int32)
    for wanted, lens, lists in ((every, got.unmasked_lens, got.unmasked_kv_ids), (some & ~every, got.masked_lens, got.masked_kv_ids)):
        n = wanted.sum(-1, dtype=torch.int32)
        assert torch.equal(lens, n.expand(2, 2, nQ))
        in_order = torch.where(wanted, ids, nK).sort(-1).values.int()
        assert torch.equal(torch.where(ids < n[..., None], lists, nK), in_order.expand(2, 2, nQ, nK))
    assert got.packed_masks is not None
    packed = got.packed_masks[:uB, :uH].reshape(uB, uH, nQ, nK, BQ, BK // 8, 1)
    bits = (packed >> torch.arange(8, dtype=torch.uint8, device=gpu)) & 1
    slots = in_order.clamp(max=nK - 1).long().view(uB, uH, nQ, nK, 1, 1).expand(uB, uH, nQ, nK, BQ, BK)
    want = tiles.transpose(3, 4).gather(3, slots)
    used = (ids < n[..., None]).view(uB, uH, nQ, nK, 1, 1)
    assert torch.equal(bits.reshape(uB, uH, nQ, nK, BQ, BK).bool() & used, want & used)


def launches_that_classify(gpu, H, nQ, BQ, Sk, BK, packing, copies):
    """One launch leaves the class bytes of the workspace as they are, three go through them."""
    lib, st, Sq = _native.load(), _native.strides, nQ * BQ
    mask = torch.zeros(1, 1, Sq, Sk, dtype=torch.bool, device=gpu).expand(1, H, Sq, Sk)
    ids = [torch.empty(1, copies, nQ, Sk // BK, dtype=torch.int32, device=gpu) for _ in range(2)]
    lens = [torch.empty(1, copies, nQ, dtype=torch.int32, device=gpu) for _ in range(2)]
    lists = [x for i, n in zip(ids, lens) for t in (i, n) for x in (t.data_ptr(), st(t.expand(1, H, *t.shape[2:]).stride()))]
    need = lib.sa_mask_classify_workspace_bytes(st(mask.stride()), 1, H, Sq, Sk, BQ, BK)
    ws = torch.full((need,), 0xAA, dtype=torch.uint8, device=gpu)
    sizes, tail = (1, H, Sq, Sk, BQ, BK), (ws.data_ptr(), need, torch.cuda.current_stream().cuda_stream)
    if packing:
        packed = torch.empty(Sq * Sk // 8, dtype=torch.uint8, device=gpu)
        rc = lib.sa_mask_classify_packed(mask.data_ptr(), st(mask.stride()), *sizes, *lists, packed.data_ptr(), st((0, 0)), *tail)
    else:
        rc = lib.sa_mask_classify(mask.data_ptr(), st(mask.stride()), *sizes, *lists, *tail)
    _native.check(rc)
    torch.cuda.synchronize()
    assert all(bool((n == 0).all()) for n in lens)
    return 1 if bool((ws == 0xAA).all()) else 3


# Where the one launch is the faster one (256 compute units): whole rounds of workgroups, and half of one where it saves the packing launch.
@pytest.mark.parametrize("nQ,BQ,Sk,BK,packing,H,copies,want", [
    (192, 128, 8192, 64, False, 1, 1, 1), (256, 128, 8192, 64, False, 1, 1, 1), (272, 128, 8192, 64, False, 1, 1, 3), (272, 128, 8192, 64, True, 1, 1, 3),
    (320, 128, 16384, 64, True, 1, 1, 3), (384, 128, 16384, 64, False, 1, 1, 1), (128, 128, 8192, 64, False, 1, 1, 3), (128, 128, 8192, 64, True, 1, 1, 1),
    (128, 128, 16384, 32, True, 32, 1, 1), (128, 128, 16384, 32, False, 32, 32, 3), (192, 128, 16384, 32, False, 32, 32, 1),
    (128, 128, 24576, 32, True, 1, 1, 3), (192, 128, 32768, 64, False, 1, 1, 3), (256, 128, 32768, 32, True, 1, 1, 1),
    (512, 64, 16384, 64, False, 1, 1, 3), (256, 64, 32768, 32, False, 1, 1, 1), (128, 64, 65536, 64, True, 1, 1, 3),
    (128, 256, 32768, 1024, True, 1, 1, 1), (128, 256, 32768, 1024, False, 1, 1, 3)])
def test_one_launch_or_three(gpu, nQ, BQ, Sk, BK, packing, H, copies, want):
    if torch.cuda.get_device_properties(0).multi_processor_count != 256:
        pytest.skip("the rule is that of 256 compute units")
    assert launches_that_classify(gpu, H, nQ, BQ, Sk, BK, packing, copies) == want
