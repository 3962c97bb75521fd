"""Row kernels at the shapes where their layout changes: rows that keep no
16-byte alignment (odd lengths, and a base pointer off by one element), rows of
a whole number of waves that is no power of two, the cached softmax's longest
rows and the streaming ones past them, and GroupNorm groups of any size walked
over many rows. Against the CPU oracle.

Tolerances: f32 rtol 1e-4 (the suite's), bf16 one rounding (2^-8 relative) of
each result beside it.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

import helion_mlir_utils as U
from oracle import restate as R
from tests.helpers import assert_close, max_rel_error, tensor, to_np

pytestmark = pytest.mark.gpu

RNG = np.random.default_rng(5)


def _rows(m: int, n: int, dtype: str, device: torch.device, offset: int, scale: float = 1.0) -> torch.Tensor:
    """A contiguous [m, n] whose first element sits `offset` elements past a
    16-byte boundary."""
    flat = tensor(RNG.normal(0, scale, m * n + offset).astype(np.float32), dtype, device)
    return flat[offset:].view(m, n)


# 64 vectors of bf16 are 512 columns, 128 are 1024; then 64-lane steps of two
# vectors a lane: 1025 takes two waves, 3001 three, 5120 five whole ones;
# 16385 and 65536 are the ends of the cached softmax's long rows (65536 f32:
# 16 vectors a lane), 65537 the first that streams.
@pytest.mark.parametrize("offset", [0, 1])
@pytest.mark.parametrize("n", [1, 7, 9, 511, 513, 1023, 1025, 3001, 5120, 16385, 24577, 49153, 65536, 65537, 100003])
@pytest.mark.parametrize("dtype", ["f32", "bf16"])
def test_softmax_row_lengths(gpu_device, n: int, dtype: str, offset: int) -> None:
    x = _rows(5, n, dtype, gpu_device, offset, 3.0)
    ref = R.softmax(to_np(x), dtype)
    got = U.softmax(x)
    assert max_rel_error(to_np(got), ref) < (1e-6 if dtype == "f32" else 2.0**-8)
    assert torch.equal(U.softmax(x, in_place=True), got)


@pytest.mark.parametrize("n", [515, 40000, 70001])
@pytest.mark.parametrize("dtype", ["f32", "bf16"])
def test_softmax_infinite_runs(gpu_device, n: int, dtype: str) -> None:
    # Runs of -inf (a masked prefix longer than any thread's first chunk), a
    # row of nothing else, +inf, NaN and the type's lowest value.
    x = RNG.normal(0, 1, (6, n)).astype(np.float32)
    x[0, : n - 1] = -np.inf
    x[1, 1:] = -np.inf
    x[2] = -np.inf
    x[3, n // 2] = np.inf
    x[4, n - 1] = np.nan
    x[5, ::2] = float(torch.finfo(torch.bfloat16).min)
    xt = tensor(x, dtype, gpu_device)
    got, ref = to_np(U.softmax(xt)), R.softmax(to_np(xt), dtype)
    assert np.array_equal(np.isnan(got), np.isnan(ref))
    assert max_rel_error(got[[0, 1, 5]], ref[[0, 1, 5]]) < (1e-6 if dtype == "f32" else 2.0**-8)


@pytest.mark.parametrize("offset", [0, 1])
@pytest.mark.parametrize(("m", "n"), [(3, 1), (5, 7), (9, 511), (4, 1025), (7, 3001), (6, 5120), (3, 12287)])
@pytest.mark.parametrize("dtype", ["f32", "bf16"])
def test_rms_norm_row_lengths(gpu_device, m: int, n: int, dtype: str, offset: int) -> None:
    x = _rows(m, n, dtype, gpu_device, offset, 2.0)
    for w_dtype in ("f32", "bf16"):
        w = _rows(1, n, w_dtype, gpu_device, offset)[0]
        ref = R.rms_norm(to_np(x), to_np(w), 1e-6, dtype)
        assert_close(to_np(U.rms_norm(x, w)), ref, 1e-4 if dtype == "f32" else 2.0**-7, 1e-5)


# (rows, groups, channels per group): groups of part of a vector, of odd
# lengths, more groups than a workgroup's units and fewer, units of several
# waves, and more rows than the GPU holds workgroups (each walks several).
@pytest.mark.parametrize("offset", [0, 1])
@pytest.mark.parametrize(("m", "groups", "gs"), [(3, 1, 1), (70, 5, 3), (9000, 32, 20), (40, 7, 160), (13, 3, 375),
                                                 (5000, 1, 3001), (300, 4, 1280), (7, 2, 5904), (11, 1, 11008)])
@pytest.mark.parametrize("dtype", ["f32", "bf16"])
def test_group_norm_group_sizes(gpu_device, m: int, groups: int, gs: int, dtype: str, offset: int) -> None:
    n = groups * gs
    x = _rows(m, n, dtype, gpu_device, offset, 2.0)
    w, b, e = (_rows(1, n, "f32", gpu_device, offset)[0] for _ in range(3))
    xs, ws, bs, es = map(to_np, (x, w, b, e))
    rtol = 1e-4 if dtype == "f32" else 2.0**-7
    # A value near 0 is a difference of products of size |w| |x| / std: its
    # absolute error is that size times f32's (bf16: the output's) rounding.
    atol = (1e-5 if dtype == "f32" else 2.0**-8) * 4
    ref = R.group_norm(xs, groups, ws, bs, 1e-5, out=dtype)
    assert_close(to_np(U.group_norm(x, groups, w, b, 1e-5)), ref, rtol, atol)
    added = R.group_norm(xs, groups, ws, bs, 1e-5, extra=es, extra_op="add", out=dtype)
    assert_close(to_np(U.group_norm(x, groups, w, b, 1e-5, torch.add, e)), added, rtol, atol)


# Short rows (lanes of a wave share them), rows of one to four vectors a lane
# (bf16: 512, 1024, 2048 columns), longer ones by 1 to 16 waves with the
# unrolled loop's remainder, few rows and many.
@pytest.mark.parametrize("offset", [0, 1])
@pytest.mark.parametrize(("m", "n"), [(3, 1), (300, 7), (1000, 65), (70, 511), (5, 1025), (9, 2047), (3, 2049),
                                     (20000, 2100), (2, 16391), (1, 70001)])
@pytest.mark.parametrize("dtype", ["f32", "bf16"])
def test_row_reductions_of_every_layout(gpu_device, m: int, n: int, dtype: str, offset: int) -> None:
    x = _rows(m, n, dtype, gpu_device, offset)
    v = _rows(1, n, "f32", gpu_device, offset)[0]
    col = _rows(n, 1, dtype, gpu_device, offset)
    xs = to_np(x).astype(np.float64)
    # f32 sums of n terms of size |x| |v|: n eps in the worst order, of which a
    # pairwise-like one shows sqrt(n); bf16 adds its rounding of the result.
    scale = np.sqrt(n) * 4
    rtol, atol = (1e-5, 2.0**-23 * np.sqrt(n) * scale) if dtype == "f32" else (2.0**-8, 2.0**-23 * n * 4)
    for got, w in ((U.row_sum(x), np.ones(n)), (U.row_dot(x, v), to_np(v)), (U.matvec(x, col), to_np(col)[:, 0])):
        assert_close(to_np(got), xs @ w.astype(np.float64)[:, None], rtol, atol)


# One chunk, two, many, up to the limit on chunks; the vector across the last
# column of every block width; one row.
@pytest.mark.parametrize("offset", [0, 1])
@pytest.mark.parametrize(("m", "n"), [(1, 3), (64, 515), (65, 513), (200, 63), (1000, 129), (5000, 257), (40000, 517),
                                     (33, 40001)])
@pytest.mark.parametrize("dtype", ["f32", "bf16"])
def test_column_sum_chunks(gpu_device, m: int, n: int, dtype: str, offset: int) -> None:
    x = _rows(m, n, dtype, gpu_device, offset)
    got = U.column_sum(x)
    assert torch.equal(got, U.column_sum(x))
    assert_close(to_np(got), to_np(x).astype(np.float64).sum(0), 1e-5, 2.0**-23 * m * 4)
