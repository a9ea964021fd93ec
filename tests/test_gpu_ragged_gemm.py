"""The GEMM kernel for rows off 16-byte boundaries (K or N not a multiple of
8, or a tensor based off one) at the edges of its tiles and K stages, against
the CPU oracle.  Integer inputs of at most 4 in magnitude make every sum exact
in fp32, so outputs and partials compare bit for bit.
"""
import numpy as np
import pytest
import torch

import oracle
from tests.test_gpu_parity import dev, host
from tests.test_gpu_random_shapes import _ints

pytestmark = pytest.mark.gpu

# 8: the smallest extents it takes; 63/65, 127/129: either side of a tile and
# of a 64-deep stage; 31/33: of a 32-deep stage (the 128 tile's)
SHAPES = [(1, 8, 9), (1, 9, 8), (65, 63, 65), (63, 65, 127), (129, 127, 33), (127, 129, 31),
          (130, 257, 72), (200, 8, 129), (70, 135, 200)]


@pytest.fixture(scope="module")
def lh():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import loom_hip
    return loom_hip


@pytest.mark.parametrize("M,N,K", SHAPES)
@pytest.mark.parametrize("tile", [64, 128])
def test_ragged_matmul_edges(lh, M, N, K, tile):
    rng = np.random.default_rng(M * 1000003 + N * 1009 + K)
    x, y = _ints(rng, (M, K)), _ints(rng, (K, N))
    ref = oracle.matmul(x, y)
    out = lh.matmul(dev(x), dev(y), tile_m=min(tile, M), tile_n=min(tile, N))
    assert np.array_equal(host(out), ref), (M, N, K, tile)


@pytest.mark.parametrize("M,N,K,tile_k", [(65, 63, 130, 65), (33, 129, 100, 33), (64, 72, 90, 8),
                                          (130, 140, 257, 64)])
def test_ragged_slabs(lh, M, N, K, tile_k):
    rng = np.random.default_rng(M + N + K)
    a, b = _ints(rng, (M, K)), _ints(rng, (K, N))
    out, parts = lh.split_k_matmul_gather(dev(a), dev(b), tile_k=tile_k)
    o_ref, p_ref = oracle.split_k_matmul_gather(a, b, 16, 16, tile_k)
    assert np.array_equal(parts.cpu().numpy(), p_ref)
    assert np.array_equal(host(out), o_ref)


@pytest.mark.parametrize("N", [64, 61])
@pytest.mark.parametrize("off", [1, 2, 3])
def test_ragged_base_addresses(lh, off, N):
    """Operands and output based at any element; what lies around them (NaN)
    neither reaches the result nor is overwritten."""
    M, K = 67, 72
    rng = np.random.default_rng(off * 100 + N)
    x, y = _ints(rng, (M, K)), _ints(rng, (K, N))

    def held(shape, a=None):
        n = int(np.prod(shape))
        buf = torch.full((n + 16,), float("nan"), dtype=torch.bfloat16, device="cuda")
        view = buf[off:off + n].view(shape)
        if a is not None:
            view.copy_(dev(a))
        return buf, view

    _, xv = held((M, K), x)
    _, yv = held((K, N), y)
    buf, out = held((M, N))
    lh.matmul(xv, yv, out)
    assert np.array_equal(host(out.clone()), oracle.matmul(x, y))
    assert torch.isnan(buf[:off]).all() and torch.isnan(buf[off + M * N:]).all()


def test_ragged_batch_beside_infinities(lh):
    """A batch whose neighbours are infinite: the loads that end at a range's
    end read the range alone."""
    M, N, K = 37, 45, 51
    rng = np.random.default_rng(5)
    x, y = _ints(rng, (M, K)), _ints(rng, (K, N))
    a = torch.full((3, M, K), float("inf"), dtype=torch.bfloat16, device="cuda")
    b = torch.full((3, K, N), float("nan"), dtype=torch.bfloat16, device="cuda")
    a[1], b[1] = dev(x), dev(y)
    assert np.array_equal(host(lh.batch_matmul(a, b)[1].contiguous()), oracle.matmul(x, y))
