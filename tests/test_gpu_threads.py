"""Calls leave the interpreter's lock to other threads while they allocate and launch."""
import sys
import threading
import time

import pytest
import torch

from sparseattention_amd import (causal_term, compute_backward_metadata, compute_mask_kernel, compute_mask_terms, select_tiling,
                                 sparse_attention, sparse_attention_backward, sparse_attention_decode, sparse_attention_tiled,
                                 workloads as W)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("call", ["classify", "terms", "forward", "forward_fresh", "tiled", "decode", "backward"])
def test_another_thread_runs_during_a_call(gpu, call):
    B, H, S, D = 1, 2, 256, 64
    q, k, v = W.qkv(B, H, S, D, torch.bfloat16, seed=3, device=gpu)
    mask = torch.ones(B, H, S, S, dtype=torch.bool, device=gpu).tril()
    md, bmd, tiling = compute_mask_kernel(mask, 128, 64), compute_backward_metadata(mask), select_tiling(mask[..., :200, :200])
    o, lse = sparse_attention(q, k, v, mask, 128, 64, md, return_lse=True)
    few, row, last = [t[:, :, :200] for t in (q, k, v)], q[:, :, :1], mask[:, :, -1:]  # (torch's own calls do let go of the lock)
    run = {
        "classify": lambda: compute_mask_kernel(mask, 128, 64),
        "terms": lambda: compute_mask_terms([causal_term()], B, H, S, S, 128, 64, device=gpu),
        "forward": lambda: sparse_attention(q, k, v, mask, 128, 64, md),
        "forward_fresh": lambda: sparse_attention(q, k, v, mask, 128, 64),
        "tiled": lambda: sparse_attention_tiled(*few, tiling),
        "decode": lambda: sparse_attention_decode(row, k, v, last, 64),
        "backward": lambda: sparse_attention_backward(o, q, k, v, o, lse, None, bmd),
    }[call]
    run()
    gate, ran = threading.Lock(), threading.Event()
    gate.acquire()
    other = threading.Thread(target=lambda: (gate.acquire(), ran.set()))
    interval = sys.getswitchinterval()
    other.start()
    time.sleep(0.05)  # (it waits at the gate)
    try:
        sys.setswitchinterval(1000)  # the interpreter itself hands the lock to nobody: only a call that lets go of it does
        gate.release()
        for _ in range(2000):
            run()
            if ran.is_set():
                break
        assert ran.is_set()
    finally:
        sys.setswitchinterval(interval)
        other.join()
    torch.cuda.synchronize()
