"""The SSD state kernel with a sequence cut into segments (few heads) and
whole (many): the chunk states against the CPU oracle's, with steps small
enough that a state is carried over many chunks.  test_segments takes headdim
and dstate to every mode of the kernel, in segments of one and two chunks and
whole; test_segment_layouts takes segments of one to five chunks, a last one
that is shorter, and carries of more than the eight slots that the joining pass
takes at a time, and checks that its cases are cut as they say.  Bars as in
tests/test_gpu_ssd.py.
"""
import numpy as np
import pytest
import torch

import oracle
from oracle import from_f16
from tests.test_gpu_f16 import dev as dev_f16, host as host_f16
from tests.test_gpu_graph import _replay_matches
from tests.test_gpu_parity import devf
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


def _segment_chunks(b, H, nc, Q, P, N):
    """Chunks per segment by the state kernel's rule (ssd.hip, segment_chunks)."""
    cap = 64 if P <= 128 else 32          # n block: the cap, dstate below it, else 32
    nb = N if N <= cap else cap if N % cap == 0 else 32
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    nseg = min(nc, cus // (b * H * (N // nb)))
    if nseg < 2:
        return nc
    cps = -(-nc // nseg)
    later = nc - cps
    return cps if later * (Q + 50) > 450 + later * (b * H * N * P) * 8 // 26667 else nc


# segments: chunks of each; with 256 CUs
LAYOUTS = [((1, 32, 16, 256, 64, 128), [4, 4, 4, 4]), ((1, 32, 15, 256, 64, 128), [4, 4, 4, 3]),
           ((1, 32, 17, 256, 64, 128), [5, 5, 5, 2]), ((1, 64, 25, 192, 32, 64), [7, 7, 7, 4]),
           ((2, 20, 16, 128, 48, 64), [3, 3, 3, 3, 3, 1]), ((1, 4, 19, 128, 128, 64), [1] * 19),
           ((3, 90, 4, 256, 64, 64), [4])]


@pytest.mark.parametrize("f16", [False, True])
@pytest.mark.parametrize("extents,layout", LAYOUTS)
def test_segment_layouts(lh, extents, layout, f16):
    b, H, nc, Q, P, N = extents
    cps = _segment_chunks(*extents)
    assert [min(cps, nc - c) for c in range(0, nc, cps)] == layout
    rng = np.random.default_rng(sum(extents))
    x, dt, A, Bm, C = _raw_inputs(rng, b, H, 1, nc * Q, P, N, dt_scale=0.001)
    what = f"layout {layout} b{b} H{H} nc{nc} Q{Q} P{P} N{N} f16={f16}"
    print("segments", what, flush=True)
    if not f16:
        _check_prologue(lh, x, dt, A, Bm, C, Q, what)
        return
    x, Bm, C = (oracle.to_f16(oracle.from_bf16(t)) for t in (x, Bm, C))
    _, _, cb, prev = lh.ssd_prologue(dev_f16(x), devf(dt), devf(A), dev_f16(Bm), dev_f16(C), Q)
    with oracle.element_type("f16"):
        _, _, cb_o, prev_o = oracle.mamba_prologue(x, dt, A, Bm, C, Q)
    cbg, cbr = from_f16(host_f16(cb)), from_f16(cb_o)
    off = int((np.abs(cbg - cbr) > 2.0 ** -10 * np.abs(cbr) + 1e-5).sum())
    assert off == 0, (what, off)
    # beside the bar: w x enters as f16 hi + lo, and steps this small leave lo on
    # f16's lowest grid (2^-24): an error of rms 2^-25 / sqrt(3) a term, times B
    # of rms 1, over the nc Q keys that a state can hold; six of these
    grid = 6 * 2.0 ** -25 / 3 ** 0.5 * (nc * Q) ** 0.5
    scale = 1e-2 * float(np.abs(prev_o).max())
    over = float((np.abs(prev.cpu().numpy() - prev_o) - 1e-3 * (np.abs(prev_o) + scale)).max())
    assert over <= grid, (what, over, grid)


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
