"""Partial results that hold an infinity: parts that a merge reads twice, or not at all, leave it what it is."""
import pytest
import torch

from sparseattention_amd import _native, compute_mask_kernel, sparse_attention, sparse_attention_decode, workloads as W

pytestmark = pytest.mark.gpu


def check(o, q, k, v, col, tol):
    s = (q.double() @ k.double().transpose(-1, -2).contiguous()) * q.shape[-1] ** -0.5
    want = torch.softmax(s, -1) @ v.double().nan_to_num(posinf=0.0)
    assert torch.isposinf(o[..., col]).all()
    o, want = o.double().clone(), want.clone()
    o[..., col] = want[..., col] = 0.0
    assert float((o - want).abs().max()) <= tol


@pytest.mark.parametrize("dtype,Sk,D,tol", [(torch.bfloat16, 4608, 128, 2e-2), (torch.float16, 4608, 64, 4e-3), (torch.float32, 1152, 64, 1e-5)])
def test_shared_lists(gpu, dtype, Sk, D, tol):
    Sq, BQ, BK = 128, 128, 64
    q, _, _ = W.qkv(1, 1, Sq, D, dtype, seed=1, device=gpu)
    _, k, v = W.qkv(1, 1, Sk, D, dtype, seed=2, device=gpu)
    v[:, :, -1, 7] = float("inf")
    assert _native.load().sa_fwd_split_workspace_bytes(1, 1, Sq, Sk, D, BQ, BK, {torch.bfloat16: 0, torch.float16: 1}.get(dtype, 2)) > 0
    mask = torch.ones(1, 1, Sq, Sk, dtype=torch.bool, device=gpu)
    check(sparse_attention(q, k, v, mask, BQ, BK, compute_mask_kernel(mask, BQ, BK)), q, k, v, 7, tol)


@pytest.mark.parametrize("splits", [8, 9, 41])
def test_decode(gpu, splits):
    Sk, D, BK = 8192, 128, 32
    q, k, v = W.qkv(1, 2, 1, D, torch.bfloat16, seed=3, device=gpu, Sk=Sk)
    v[:, :, -1, 7] = float("inf")
    mask = torch.ones(1, 2, 1, Sk, dtype=torch.bool, device=gpu)
    check(sparse_attention_decode(q, k, v, mask, BK, compute_mask_kernel(mask, 1, BK), num_splits=splits), q, k, v, 7, 2e-2)
