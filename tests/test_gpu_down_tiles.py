"""The down-projection of weights without blocks at the edges of its tiles (32
and 64 rows and outputs, an eighth of K a wave): every element one of the two
bf16 neighbours of the float64 product up to fp32 accumulation."""
import numpy as np
import pytest
import torch

from oracle import attention as oa
from tests.helpers import neighbour_of_exact, to_np

pytestmark = pytest.mark.gpu


def _problem(device, K, N, B, L, n):
    gen = torch.Generator(device=device).manual_seed(K + N + n)
    x = torch.randn(B, L, K, generator=gen, device=device).to(torch.bfloat16)
    w = (torch.randn(N, K, generator=gen, device=device) / K ** 0.5).to(torch.bfloat16)
    return x, w, torch.randperm(L, generator=gen, device=device)[:n].contiguous()


def _check(got, x, w, rows):
    idx = rows.cpu().numpy()
    exact = oa.down_project(to_np(x), to_np(w), idx, bf16_boundaries=False)
    terms = oa.down_project(np.abs(to_np(x)), np.abs(to_np(w)), idx, bf16_boundaries=False)
    neighbour_of_exact(to_np(got), exact, exact_rounded(exact), terms)


def exact_rounded(x):
    return to_np(torch.from_numpy(x).to(torch.bfloat16))


@pytest.mark.parametrize('K,N,B,n', [(32, 16, 1, 1), (160, 48, 2, 33), (1056, 272, 3, 31), (4096, 256, 1, 64),
                                     (5120, 384, 4, 300), (96, 1040, 1, 700), (4096, 64, 1, 4),
                                     (4096, 64, 5, 1), (1056, 48, 1, 36), (1056, 48, 1, 37)])
def test_tile_edges(device, K, N, B, n):
    from slimkv_amd import kernels
    x, w, rows = _problem(device, K, N, B, n + 9, n)
    _check(kernels.down_project(x, w, rows), x, w, rows)


@pytest.mark.parametrize('sizes', [((4096, 256, 64), (4096, 320, 64)), ((256, 64, 40), (256, 1024, 900))])
def test_pair_equals_single_launches(device, sizes):
    from slimkv_amd import kernels
    problems = [_problem(device, K, N, 2, n + 5, n) for K, N, n in sizes]
    pair = kernels.down_project_pair(*({'x': x, 'weight': w, 'rows': r} for x, w, r in problems))
    for got, (x, w, r) in zip(pair, problems):
        assert torch.equal(got, kernels.down_project(x, w, r))
