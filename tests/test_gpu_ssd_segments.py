"""The SSD state kernel with a sequence cut into segments (few heads) and
whole (many): the chunk states against the CPU oracle's, with steps small
enough that a state is carried over many chunks.  Chunk counts leave the last
segment whole, short and of one chunk; headdim and dstate reach every mode of
the kernel.  Bars as in tests/test_gpu_ssd.py.
"""
import numpy as np
import pytest
import torch

from tests.test_gpu_graph import _replay_matches
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


def test_segments_captured(lh):
    g = torch.Generator(device="cuda").manual_seed(3)
    b, H, nc, Q, P, N = 1, 4, 16, 256, 64, 128
    L = nc * Q
    x = torch.randn(b, H, L, P, device="cuda", generator=g).to(torch.bfloat16)
    dt = torch.rand(b, H, L, device="cuda", generator=g) * 0.01
    A = -torch.rand(H, device="cuda", generator=g)
    Bm, C = (torch.randn(b, 1, L, N, device="cuda", generator=g).to(torch.bfloat16) for _ in "BC")
    _, dA, cb, prev = lh.ssd_prologue(x, dt, A, Bm, C, Q)
    _replay_matches("ssd segments", lambda: lh.ssd_prologue(
        x, dt, A, Bm, C, Q, dA_cumsum=dA, cb=cb, prev_states_T=prev), [dA, cb, prev])
