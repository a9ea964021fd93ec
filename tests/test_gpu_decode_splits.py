"""flash_decode's combine at every split count its forms divide at (8, 16 and
the chunks of 8 splits per thread group), for few and many rows, and both
kernels of K rows off 16-byte boundaries (splits up to and above 512 keys);
against the CPU oracle, out and partials, at decode's bars.
"""
import math

import numpy as np
import pytest
import torch

import oracle
from oracle import from_bf16, to_bf16
from tests.conftest import assert_close
from tests.test_gpu_parity import ATTN_TOL, dev, host, rng_bf16

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def lh():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import loom_hip
    return loom_hip


def _check(lh, B, H, D, S, tile_s):
    rng = np.random.default_rng(B + 3 * H + 5 * D + S + tile_s)
    k, v, q = rng_bf16(rng, (B, D, S)), rng_bf16(rng, (B, S, D)), rng_bf16(rng, (B, H, D))
    print(f"decode B{B} H{H} D{D} S{S} tile_s {tile_s}", flush=True)
    ref, lse, o = oracle.flash_decode(k, v, q, 1 / math.sqrt(D), 1, tile_s, min(64, tile_s))
    out, glse, go = lh.flash_decode(dev(k), dev(v), dev(q), tile_s=tile_s, return_partials=True)
    what = f"B{B} H{H} D{D} S{S} tile_s {tile_s}"
    assert_close(from_bf16(host(out)), from_bf16(ref), **ATTN_TOL, what=what)
    assert_close(glse.cpu().numpy(), lse, atol=1e-2, rtol=1e-3, what=what + " lse")
    assert_close(go.cpu().numpy(), o, atol=2e-2, rtol=1e-2, what=what + " o")


@pytest.mark.parametrize("D", [8, 64, 72, 128, 256])
@pytest.mark.parametrize("ns", [8, 9, 16, 17, 65, 130])
def test_split_counts(lh, D, ns):
    _check(lh, 2, 5, D, 16 * ns - 8, 16)


@pytest.mark.parametrize("ns", [9, 16, 17])
def test_split_counts_many_rows(lh, ns):
    _check(lh, 33, 32, 128, 32 * ns, 32)


@pytest.mark.parametrize("S,tile_s", [(1031, 512), (1031, 513), (1030, 512), (2047, 1024),
                                      (1601, 1600), (67, 67)])
@pytest.mark.parametrize("D,H", [(64, 9), (128, 32)])
def test_ragged_keys_split_lengths(lh, S, tile_s, D, H):
    _check(lh, 2, H, D, S, tile_s)


# hidden keys by 32-key halves of a 64-key block: a half's first block, both of
# its first two, the other half's; the rest of each split is finite
@pytest.mark.parametrize("hidden", [((0, 32),), ((32, 64),), ((0, 32), (64, 96)),
                                    ((32, 64), (192, 224))])
@pytest.mark.parametrize("S", [389, 392])
@pytest.mark.parametrize("D,H", [(64, 9), (128, 20), (128, 40), (256, 20)])
def test_infinite_scores_of_some_heads(lh, hidden, S, D, H):
    """Keys whose score is -inf for the odd heads (a k of the type's lowest
    value, beyond fp32 against their q) and ordinary for the even ones, with
    finite scores far below zero elsewhere."""
    rng = np.random.default_rng(S + D + H)
    k, v, q = (rng.standard_normal(s).astype(np.float32)
               for s in ((1, D, S), (1, S, D), (1, H, D)))
    q[:, 0::2, 0], q[:, 1::2, 0] = 0.0, 8.0
    k[:, 0, :] = -600.0
    for a, b in hidden:
        k[:, 0, a:b] = -3.0e38
    k, v, q = to_bf16(k), to_bf16(v), to_bf16(q)
    print(f"decode -inf H{H} D{D} S{S} hidden {hidden}", flush=True)
    got = from_bf16(host(lh.flash_decode(dev(k), dev(v), dev(q), tile_s=192)))
    s = (from_bf16(q)[0].astype(np.float64) @ from_bf16(k)[0].astype(np.float64)) / math.sqrt(D)
    p = np.exp(s - s.max(-1, keepdims=True))
    ref = (p / p.sum(-1, keepdims=True)) @ from_bf16(v)[0].astype(np.float64)
    assert_close(got[0], ref, **ATTN_TOL, what=f"hidden {hidden} H{H} D{D} S{S}")
