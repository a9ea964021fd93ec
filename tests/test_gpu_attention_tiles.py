"""The attention kernels on both sides of the rule that picks the query tile of
a call that leaves it free (small grids: 64 rows whose keys two waves share),
and bound tiles (64 .. 256), which run as bound on any grid.  Sampled heads
against the CPU oracle, at attention's bar (tests/test_gpu_parity.py).
"""
import math

import numpy as np
import pytest
import torch

import oracle
from oracle import from_bf16, from_f16, to_bf16, to_f16
from tests.conftest import assert_close
from tests.test_gpu_parity import ATTN_TOL, dev, host, rng_bf16

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def lh():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import loom_hip
    return loom_hip


def _check(lh, BH, Sq, Skv, D, causal, tile_m, heads):
    """In bf16 and in f16: each type has its own build of every tile."""
    h = list(heads)
    for name, to, back, dtype in (("bf16", to_bf16, from_bf16, torch.bfloat16),
                                  ("f16", to_f16, from_f16, torch.float16)):
        rng = np.random.default_rng(BH + 7 * Sq + Skv + D)
        k, v, q = (to(rng.standard_normal(s, dtype=np.float32))
                   for s in ((BH, D, Skv), (BH, Skv, D), (BH, Sq, D)))
        what = f"{name} tile {tile_m} BH{BH} Sq{Sq} Skv{Skv} D{D} {causal}"
        print("attention", what, flush=True)
        got = lh.attention(*(dev(t).view(dtype) for t in (k, v, q)), causal=causal, tile_m=tile_m)
        assert got.dtype == dtype
        with oracle.element_type(name):
            ref = back(oracle.attention(k[h], v[h], q[h], 1 / math.sqrt(D), causal, 1, 64, 64))
        assert_close(back(host(got))[h], ref, **ATTN_TOL, what=what)


# more than four workgroups of 64 rows per CU of 256
@pytest.mark.parametrize("D,tile_m", [(64, 64), (64, 128), (64, 192), (64, 256), (72, 128),
                                      (128, 64), (128, 128), (128, 192), (128, 256), (200, 128)])
@pytest.mark.parametrize("Sq,Skv,causal", [(270, 270, True), (264, 264, True), (260, 100, False),
                                           (257, 61, False)])
def test_large_grids_run_the_bound_tile(lh, D, tile_m, Sq, Skv, causal):
    _check(lh, 216, Sq, Skv, D, causal, tile_m, (0, 101, 215))


# one to four workgroups of 64 rows per CU, and the rule's edges (256, 512 and
# 1024 of them on 256 CUs)
@pytest.mark.parametrize("BH,Sq,Skv,D,causal", [
    (3, 300, 300, 128, True), (64, 256, 256, 128, True), (128, 256, 264, 128, False),
    (129, 256, 264, 128, False), (256, 250, 250, 64, True), (129, 256, 40, 64, False),
    (64, 256, 72, 256, False), (2, 130, 33, 128, False), (2, 64, 32, 128, False),
    (2, 70, 31, 64, False), (1, 1, 1, 128, False), (2, 96, 96, 256, True)])
def test_small_grids(lh, BH, Sq, Skv, D, causal):
    for tile_m in (None, min(256, Sq)):
        _check(lh, BH, Sq, Skv, D, causal, tile_m, range(0, BH, max(1, BH // 3)))


@pytest.mark.parametrize("D,tile_m", [(64, 128), (64, 192), (64, 256), (96, 128), (96, 192),
                                      (96, 256), (128, 64), (128, 128), (128, 192), (128, 256),
                                      (256, 64), (256, 128)])
@pytest.mark.parametrize("Skv", [256, 61])
def test_bound_tile_on_any_grid(lh, D, tile_m, Skv):
    """A bound tile runs as bound whatever the grid: the heads of a small call
    are bit for bit those of a large one, and tiles of more than 64 rows, which
    sum a row's keys in one order, agree with each other."""
    rng = np.random.default_rng(D + tile_m)
    BH, Sq = 300, 256
    k, v, q = (dev(rng_bf16(rng, s)) for s in ((BH, D, Skv), (BH, Skv, D), (BH, Sq, D)))
    print(f"attention bound tile {tile_m} D{D} Skv{Skv}", flush=True)
    large = lh.attention(k, v, q, tile_m=tile_m)
    small = lh.attention(k[:2].contiguous(), v[:2].contiguous(), q[:2].contiguous(), tile_m=tile_m)
    assert torch.equal(small, large[:2])
    if tile_m > 64:
        assert torch.equal(large, lh.attention(k, v, q, tile_m=128))


@pytest.mark.parametrize("hidden", [(32, 64), (0, 32), (0, 64), (64, 128)])
def test_halves_of_infinite_scores(lh, hidden):
    """Keys of -inf score (an infinite k against a positive q) over one half
    of a stage or all of it, and finite scores far below zero elsewhere: the
    half's base is set by its first finite score."""
    D, S = 64, 160
    rng = np.random.default_rng(9)
    q = np.zeros((1, 70, D), np.float32)
    q[:, :, 0] = 8.0
    q[:, :, 1:] = rng.standard_normal((1, 70, D - 1))
    k = rng.standard_normal((1, D, S)).astype(np.float32)
    k[:, 0, :] = -600.0
    k[:, 0, hidden[0]:hidden[1]] = -np.inf
    v = rng.standard_normal((1, S, D)).astype(np.float32)
    k, v, q = to_bf16(k), to_bf16(v), to_bf16(q)
    got = from_bf16(host(lh.attention(dev(k), dev(v), dev(q))))
    s = (from_bf16(q)[0].astype(np.float64) @ from_bf16(k)[0].astype(np.float64)) / math.sqrt(D)
    p = np.exp(s - s.max(-1, keepdims=True))
    ref = (p / p.sum(-1, keepdims=True)) @ from_bf16(v)[0].astype(np.float64)
    # every score shares the offset -600 * 8 / 8 = -600 log-units; q is scaled
    # and rounded to bf16 once, which moves a score by up to 2^-9 of its terms'
    # sum (about 600 * 2^-9 = 1.2 common to all keys, and 2^-9 * sum |q k| / 8
    # between them): the common part cancels
    assert_close(got[0], ref, atol=3e-2, rtol=2e-2, what=f"hidden {hidden}")


def test_nan_reaches_the_row(lh):
    """A NaN in either half of the keys makes every row NaN."""
    rng = np.random.default_rng(10)
    for key in (5, 40, 100):
        k, v, q = rng_bf16(rng, (1, 64, 128)), rng_bf16(rng, (1, 128, 64)), rng_bf16(rng, (1, 64, 64))
        kt = dev(k)
        kt[0, 3, key] = float("nan")
        assert torch.isnan(lh.attention(kt, dev(v), dev(q))).all(), key


# head dims whose products run over 96 of the 128 staged columns, at each query
# tile, and 104 beside them; V rows of odd pieces (61 keys) take K by registers
@pytest.mark.parametrize("D,tile_m", [(80, 64), (96, 64), (96, 128), (80, 192), (88, 256),
                                      (96, 256), (104, 256)])
@pytest.mark.parametrize("BH,Sq,Skv,causal", [(216, 270, 270, True), (216, 257, 61, False),
                                              (24, 130, 130, True)])
def test_heads_of_up_to_96(lh, D, tile_m, BH, Sq, Skv, causal):
    _check(lh, BH, Sq, Skv, D, causal, min(tile_m, Sq), (0, BH // 2, BH - 1))
