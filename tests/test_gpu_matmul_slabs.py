"""matmul's K slabs (a long K over few output tiles, tiles left to the
library) against the CPU oracle and against one pass, and the rule's edges.
Integer inputs of at most 4 in magnitude keep every sum exact below 2^24
(16 K <= 2^17), so both ways give the same bits."""
import numpy as np
import pytest
import torch

import oracle
from tests.test_gpu_graph import _replay_matches
from tests.test_gpu_parity import dev, host
from tests.test_gpu_random_shapes import _ints


@pytest.fixture(scope="module")
def lh():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import loom_hip
    return loom_hip


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(1, 8, 3200), (40, 576, 4096), (64, 64, 8192), (65, 129, 3328),
                                   (33, 47, 1700), (200, 175, 2229), (1, 1, 2000), (16, 1000, 3208),
                                   (640, 640, 3200)])
def test_matmul_slabs(lh, M, N, K):
    assert lh._slabs(M, N, K)
    rng = np.random.default_rng(M + N + K)
    x, y = _ints(rng, (M, K)), _ints(rng, (K, N))
    ref = oracle.matmul(x, y)
    got = lh.matmul(dev(x), dev(y))
    assert np.array_equal(host(got), ref)
    one = lh.matmul(dev(x), dev(y), tile_k=1)      # a bound tile: one pass
    assert torch.equal(got, one)
    out = torch.empty_like(got)
    assert lh.matmul(dev(x), dev(y), out) is out and torch.equal(out, got)


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(40, 576, 4096), (33, 47, 1700)])
def test_slabs_captured(lh, M, N, K):
    """The partials' allocation and both launches inside a graph."""
    rng = np.random.default_rng(M)
    x, y = dev(_ints(rng, (M, K))), dev(_ints(rng, (K, N)))
    out = torch.empty(M, N, dtype=torch.bfloat16, device="cuda")
    _replay_matches(f"matmul slabs {M}x{N}x{K}", lambda: lh.matmul(x, y, out), [out])


def test_rule():
    import loom_hip as lh
    for M, N, K in [(1024, 1024, 1024), (128, 128, 1024), (2048, 2048, 1 << 20), (64, 64, 255),
                    (64, 64, 3192), (33, 47, 1699), (1 << 20, 8, 4096)]:
        assert lh._slabs(M, N, K) == 0, (M, N, K)
    rng = np.random.default_rng(0)
    for _ in range(3000):
        M, N, K = (int(v) for v in np.exp(rng.uniform(0, np.log(1 << 15), 3)))
        tk = lh._slabs(M, N, K)
        if tk:
            S = -(-K // tk)
            assert tk % 64 == 0 and 256 <= tk < K and 2 <= S <= 16
            assert S * -(-M // 64) * -(-N // 64) <= 256 and 4 * S * M * N <= 4 << 20
