"""K ranges that are not a whole number of the pipelined GEMM kernel's rounds
(4 or 8 stages of 32): fewer stages than a round, one more or one fewer, a
partial last stage of 8, 16 or 24 columns, and slabs that end so.  Integer
inputs keep every sum exact, so results compare bit for bit with the CPU
oracle.
"""
import numpy as np
import pytest
import torch

import oracle
from tests.test_gpu_parity import dev, host
from tests.test_gpu_random_shapes import _ints

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def lh():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import loom_hip
    return loom_hip


@pytest.mark.parametrize("tile", [64, 128, 256])
@pytest.mark.parametrize("K", [8, 24, 32, 40, 96, 128, 136, 160, 248, 256, 264, 416, 520])
def test_matmul_any_k(lh, tile, K):
    M, N = 270, 264
    rng = np.random.default_rng(K + tile)
    x, y = _ints(rng, (M, K)), _ints(rng, (K, N))
    out = lh.matmul(dev(x), dev(y), tile_m=tile, tile_n=tile)
    assert np.array_equal(host(out), oracle.matmul(x, y)), (K, tile)


@pytest.mark.parametrize("tile", [64, 128])
@pytest.mark.parametrize("K,tile_k", [(520, 256), (600, 200), (1040, 520), (72, 8)])
def test_slabs_any_k(lh, tile, K, tile_k):
    M, N = 136, 144
    rng = np.random.default_rng(K + tile_k)
    a, b = _ints(rng, (M, K)), _ints(rng, (K, N))
    out, parts = lh.split_k_matmul_gather(dev(a), dev(b), tile_m=tile, tile_n=tile, tile_k=tile_k)
    o_ref, p_ref = oracle.split_k_matmul_gather(a, b, 16, 16, tile_k)
    assert np.array_equal(parts.cpu().numpy(), p_ref)
    assert np.array_equal(host(out), o_ref)


def test_partial_stage_beside_infinities(lh):
    """Infinite neighbours of a batch's last, partial K stage stay out of it."""
    M, N, K = 40, 48, 56
    rng = np.random.default_rng(6)
    x, y = _ints(rng, (M, K)), _ints(rng, (K, N))
    a = torch.full((3, M, K), float("inf"), dtype=torch.bfloat16, device="cuda")
    b = torch.full((3, K, N), float("nan"), dtype=torch.bfloat16, device="cuda")
    a[1], b[1] = dev(x), dev(y)
    assert np.array_equal(host(lh.batch_matmul(a, b)[1].contiguous()), oracle.matmul(x, y))
