"""The short way of a well-formed call (loom_hip._plan, _prologue_plan) accepts
exactly the signatures that the full checks accept, and gives the same
extents, tiles and output shapes (CPU only: signatures are types and shapes)."""
import itertools
import weakref

import numpy as np
import pytest
import torch

import loom_hip as lh

bf, f16, f32 = torch.bfloat16, torch.float16, torch.float32


def _meta(dtype, shape):
    return torch.empty(shape, dtype=dtype, device="meta")


def _full(func, tensors, given):
    """Extents, tiles, type and output shape by the full checks."""
    e, _ = lh._elt(tensors[1 if func == "helion_mamba2_chunk_scan_kernel" else 0])
    dims = lh._dims_of(func, tensors)
    spec = lh._SPECS[func](*dims)
    side = f32 if e == bf else f16
    for t, (name, kind, shape) in zip(tensors, spec):
        lh._check_form(t, name, e if kind == "e" else side, shape)
    return tuple(dims), tuple(lh._tiles(func, dims, **given)), e, tuple(spec[-1][2])


CALLS = {
    "matmul": ([(64, 32), (32, 48)], ("tile_m", "tile_n", "tile_k")),
    "batch_matmul": ([(2, 64, 32), (2, 32, 48)], ("tile_b", "tile_m", "tile_n", "tile_k")),
    "split_k_matmul_gather": ([(64, 512), (512, 48)], ("tile_m", "tile_n", "tile_k")),
    "attention": ([(2, 64, 100), (2, 100, 64), (2, 90, 64)], ("tile_b", "tile_m", "tile_n")),
    "flash_decode": ([(2, 64, 100), (2, 100, 64), (2, 9, 64)], ("tile_b", "tile_s", "tile_n")),
    "helion_mamba2_chunk_scan_kernel": (
        [(1, 2, 1, 64, 64), (1, 4, 128, 32), (1, 4, 2, 64), (1, 4, 2, 64), (1, 1, 128, 64), (4,),
         (1, 2, 4, 64, 32)], ("tile_b", "tile_h", "tile_c", "tile_m", "tile_n", "tile_k")),
}


def _variants(shapes):
    """The signature itself, each extent of each input one off, a dimension
    more or fewer, and every choice of one input's type."""
    yield shapes, None
    for i, s in enumerate(shapes):
        for d in range(len(s)):
            yield [t if j != i else s[:d] + (s[d] + 1,) + s[d + 1:] for j, t in enumerate(shapes)], None
        yield [t if j != i else s[:-1] for j, t in enumerate(shapes)], None
        yield [t if j != i else (1,) + s for j, t in enumerate(shapes)], None
        for dt in (bf, f16, f32):
            yield shapes, (i, dt)


@pytest.mark.parametrize("func", CALLS)
@pytest.mark.parametrize("base", [bf, f16, f32])
@pytest.mark.parametrize("tile", [None, 16])
def test_plans_match_the_full_checks(func, base, tile):
    shapes0, symbols = CALLS[func]
    given = {s: (1 if s in ("tile_b", "tile_h", "tile_c") else tile) if tile else None
             for s in symbols}
    accepted = 0
    for shapes, change in _variants(shapes0):
        sides = {2, 3, 5, 6} if func.startswith("helion") else set()
        types = [f32 if i in sides and base == bf else base for i in range(len(shapes))]
        if change:
            types[change[0]] = change[1]
        tensors = [_meta(t, s) for t, s in zip(types, shapes)]
        sig = tuple(itertools.chain.from_iterable((t.dtype, t.shape) for t in tensors))
        plan = lh._plan(func, sig, tuple(given.items()))
        try:
            want = _full(func, tensors, given)
        except (ValueError, TypeError, RuntimeError):
            want = None
        assert (plan is None) == (want is None), (func, shapes, types)
        if tile is None:      # a call that gives no tile
            assert lh._plan(func, sig, ()) == plan
        if plan:
            accepted += 1
            assert plan[2:] == want
            assert plan[1] == "loom_hip_" + func + ("_f16" if want[2] == f16 else "")
    assert accepted or base == f32


@pytest.mark.parametrize("base", [bf, f16, f32])
def test_prologue_plans(base):
    shapes0 = [(1, 4, 128, 32), (1, 4, 128), (4,), (1, 2, 128, 64), (1, 2, 128, 64)]
    accepted = 0
    for (shapes, change), Q in itertools.product(_variants(shapes0), (64, 128, 48, 0, -64)):
        types = [base, f32, f32, base, base]
        if change:
            types[change[0]] = change[1]
        tensors = [_meta(t, s) for t, s in zip(types, shapes)]
        sig = tuple(itertools.chain.from_iterable((t.dtype, t.shape) for t in tensors))
        plan = lh._prologue_plan(sig, Q)
        try:
            lh.ssd_prologue(*tensors, Q)
            want = "accepted"
        except (ValueError, TypeError) as err:
            want = str(err)
        # the full checks accept the form, and stop at the device
        assert (plan is not None) == ("ROCm device" in want), (shapes, types, Q, want)
        if plan:
            accepted += 1
            b, H, L, P = shapes[0]
            G, N = shapes[3][1], shapes[3][3]
            assert plan[2] == (b, L // Q, H, G, Q, P, N)
            assert [s for _, s in plan[3]] == [(b, H, L // Q, Q), (b, L // Q, G, Q, Q),
                                               (b, L // Q, H, N, P)]
    assert accepted or base == f32


# either side of each line: 64-row workgroups per CU of 256 (one above D 128,
# two, four when causal), and short Sq
@pytest.mark.parametrize("BH,Sq,D,causal,want", [
    (8, 4096, 128, False, 64), (8, 4097, 128, False, 256), (16, 4096, 64, True, 64),
    (16, 4097, 64, True, 256), (4, 4096, 256, True, 64), (4, 4097, 136, False, 128),
    (1, 40, 64, False, 40), (1, 1000, 80, True, 64), (600, 40, 128, False, 40),
    (600, 100, 128, False, 64), (600, 200, 128, False, 192), (600, 40, 128, True, 40),
    (171, 192, 64, False, 192), (170, 192, 64, False, 64), (1 << 40, 1 << 40, 128, False, 256)])
def test_free_query_tile(BH, Sq, D, causal, want):
    t = dict(tile_b=None, tile_m=None, tile_n=None)
    dims = BH, Sq, Sq, D
    assert lh._tiles("attention", dims, causal, **t)[1] == want
    sig = (bf, (BH, D, Sq), bf, (BH, Sq, D), bf, (BH, Sq, D))
    assert lh._plan("attention", sig, tuple(t.items()), causal)[3][1] == want
    for tile in (16, min(128, Sq), Sq):      # a bound one stays
        assert lh._tiles("attention", dims, causal, **{**t, "tile_m": tile})[1] == tile


class _OnDevice(torch.Tensor):
    """A tensor without memory that says it lies on device 0, as _enter asks."""

    def get_device(self):
        return 0


def _on_device(dtype, shape):
    return _meta(dtype, shape).as_subclass(_OnDevice)


def test_plans_hold_the_value_of_a_tile(monkeypatch):
    """A tile given as an object whose value changes: each call takes the value
    it has then, and the plan keeps no reference to the object."""
    monkeypatch.setattr(lh, "_raw_stream", lambda i: 0)
    ab = _on_device(bf, (64, 512)), _on_device(bf, (512, 48))

    def tiles(tk):
        return lh._enter("split_k_matmul_gather", ab, None,
                         (("tile_m", 64), ("tile_n", None), ("tile_k", tk)))[0][3]
    tk = torch.tensor(128)
    assert tiles(tk) == (64, 48, 128)
    tk.fill_(256)
    assert tiles(tk) == (64, 48, 256)
    dead = weakref.ref(tk)
    del tk
    assert dead() is None
    for value in (np.int64(64), 64.0, 64):
        assert tiles(value) == (64, 48, 64)
    for value in (float("inf"), float("nan"), "x", (1,)):     # the full checks say what is wrong
        assert lh._enter("matmul", ab, None, (("tile_m", value),)) is None


def test_prologue_chunk_size_of_another_type(monkeypatch):
    """A chunk size that is no int goes the full way and leaves the int's own
    plan alone, though the two compare and hash equal."""
    monkeypatch.setattr(lh, "_raw_stream", lambda i: 0)
    ins = [_on_device(t, s) for t, s in zip(
        (bf, f32, f32, bf, bf), [(1, 4, 96, 32), (1, 4, 96), (4,), (1, 2, 96, 64), (1, 2, 96, 64)])]
    for Q in (np.int64(48), 48.0, torch.tensor(48)):
        assert lh._enter_prologue(ins, (None,) * 3, Q) is None
    assert lh._enter_prologue(ins, (None,) * 3, 48)[0][2] == (1, 2, 4, 2, 48, 32, 64)


def test_cpu_calls_take_the_full_checks():
    assert lh._enter("matmul", (torch.zeros(4, 4, dtype=bf), torch.zeros(4, 4, dtype=bf)), None,
                     ()) is None
    assert lh._enter("matmul", (None, 3), None, ()) is None
