"""The SSD state kernel with a sequence cut into segments (few heads) and
whole (many): the chunk states against the CPU oracle's, with steps small
enough that a state is carried over many chunks.  Chunk counts leave the last
segment whole, short and of one chunk; headdim and dstate reach every mode of
the kernel.  Bars as in tests/test_gpu_ssd.py.
"""
import numpy as np
import pytest
import torch

from tests.test_gpu_ssd import _check_prologue, _raw_inputs

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def lh():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import loom_hip
    return loom_hip


@pytest.mark.parametrize("P,N,Q", [(64, 64, 256), (64, 128, 128), (64, 32, 192), (32, 64, 256),
                                   (48, 64, 128), (128, 64, 128), (256, 32, 64)])
@pytest.mark.parametrize("b,H,nc", [(1, 2, 2), (1, 2, 9), (2, 40, 5), (2, 40, 6), (3, 90, 4)])
def test_segments(lh, P, N, Q, b, H, nc):
    if b * H * nc * Q * P * N > 3e9:
        pytest.skip("oracle time")
    rng = np.random.default_rng(P + N + Q + H + nc)
    x, dt, A, Bm, C = _raw_inputs(rng, b, H, 1, nc * Q, P, N, dt_scale=0.01)
    print(f"segments b{b} H{H} nc{nc} Q{Q} P{P} N{N}", flush=True)
    _check_prologue(lh, x, dt, A, Bm, C, Q, f"b{b} H{H} nc{nc} Q{Q} P{P} N{N}")
