"""Merge of a decode's partial results: few parts and many take different kernels (nine and more: eight parts side by side).

A part's rows are float32; weights, sums and order of addition differ by float32 roundings (2^-24 each, at most 256 parts)
below half a step of the 16-bit result, which may land one step away (2^-8 in bf16, 2^-11 in fp16, of the value)."""
import pytest
import torch

from sparseattention_amd import compute_mask_kernel, sparse_attention_decode, workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D,dtype", [(64, torch.bfloat16), (128, torch.bfloat16), (128, torch.float16)])
@pytest.mark.parametrize("Sq", [1, 3, 32])
def test_every_number_of_parts(gpu, Sq, D, dtype):
    B, H, Sk, BK = 1, 3, 8192, 32
    q, k, v = W.qkv(B, H, Sq, D, dtype, seed=Sq, device=gpu, Sk=Sk)
    mask = torch.zeros(B, H, Sq, Sk, dtype=torch.bool, device=gpu)
    mask[:, 0, :, :6000] = True
    mask[:, 1, :, ::97] = True
    mask[:, 2, :, 64:70] = True  # (one chunk: all parts but one are empty)
    if Sq > 1:
        mask[:, :, 1] = False  # a row without a key in any part
    md = compute_mask_kernel(mask, Sq, BK)
    s = q.double() @ k.double().transpose(-1, -2).contiguous() / D ** 0.5
    s = s.masked_fill(~mask, float("-inf"))
    lse64 = torch.logsumexp(s, -1)
    # q is scaled and rounded to 16 bits, P too: a score is off by a rounding of every product at most, a row sum by one of P
    size = (q.double().abs() @ k.double().abs().transpose(-1, -2).contiguous() / D ** 0.5).masked_fill(~mask, 0).amax(-1)
    step = 2.0 ** (-8 if dtype == torch.bfloat16 else -11)
    want = None
    for n in (8, 9, 16, 33, 64, 65, 255, 256):
        o, lse = sparse_attention_decode(q, k, v, mask, BK, md, num_splits=n, return_lse=True)
        torch.cuda.synchronize()
        assert torch.equal(torch.isinf(lse), torch.isinf(lse64))
        on = ~torch.isinf(lse)
        assert ((lse.double() - lse64).abs()[on] <= (step * (1 + size) + 1e-5)[on]).all()
        if want is None:
            want = o  # (eight parts: the other kernel)
        # parts cut elsewhere round P against other reference values: half a step on each side, and the result's own
        torch.testing.assert_close(o.float(), want.float(), rtol=2 * step, atol=2 * step * v.abs().max().item())
