"""That bench.py's cases run: the names they import exist (no GPU), and forward and backward at a small size."""
import ast
import importlib
import inspect

import pytest
import torch

import bench


def test_imported_names_exist():
    for node in ast.walk(ast.parse(inspect.getsource(bench))):
        if isinstance(node, ast.ImportFrom) and node.module and node.module.split(".")[0] in ("sparseattention_amd", "oracle"):
            module = importlib.import_module(node.module)
            for alias in node.names:
                assert hasattr(module, alias.name) or importlib.util.find_spec(f"{node.module}.{alias.name}"), alias.name


@pytest.mark.gpu
@pytest.mark.parametrize("S,p,schedule,kernel", [(1024, None, None, "sparse_fwd_kernel"), (1024, 0.9, None, "sparse_fwd_c32_kernel"),
                                                 (1024, 0.9, "pairs", "sparse_fwd_kernel")])
def test_forward_case(gpu, S, p, schedule, kernel):
    from sparseattention_amd import workloads as W

    q, k, v = W.qkv(1, 2, S, 128, torch.bfloat16, seed=0, device=gpu)
    mask = W.causal_mask(S, gpu) if p is None else W.random_block_mask(S, 128, p, seed=1, device=gpu)
    row = bench.forward_case("small", mask, q, k, v, 2, 1, schedule=schedule)
    assert row["_kernel"] == kernel and row["kernel_ms"] > 0
    assert 0 < row["_useful_flop"] <= row["_executed_flop"]


@pytest.mark.gpu
@pytest.mark.parametrize("H,kernel", [(2, "sparse_bwd_kernel (+"), (64, "sparse_bwd_keys_kernel, sparse_bwd_queries_kernel (+")])
def test_backward_case(gpu, monkeypatch, H, kernel):
    from sparseattention_amd import workloads as W

    B, S = 1, 1024
    for name, value in (("B", B), ("H", H), ("S", S)):
        monkeypatch.setattr(bench, name, value)
    row = bench.backward_case(*W.qkv(B, H, S, 128, torch.bfloat16, seed=0, device=gpu), 2, 1)
    assert row["roofline"]["kernel"].startswith(kernel)
    # five products per tile where dS is stored, eight where it is made anew
    tiles = row["executed_tiles_per_plane"]
    flop = 2 * 128 * 64 * 128 * B * H * (tiles["by_query"] + 4 * tiles["by_key"] if H == 64 else 3 * tiles["by_query"] + 5 * tiles["by_key"])
    assert row["executed_tflops"] == pytest.approx(flop / (row["kernel_ms"] * 1e-3) / 1e12, rel=0.02, abs=0.1)
