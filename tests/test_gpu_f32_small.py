"""Small f32 products, whose 32 x 32 tiles split K inside the workgroup: edges of
the tiles, K of one step past a wave's share up to many, each operand stored
either way at any alignment, batches and epilogues. Against the f64
product, with the memory around the operands filled with NaN.

Tolerance: f32 sums of K products in any order stay within K * 2^-24 * sum |a b|
of the exact one (doubled for the products' own rounding).
"""

from __future__ import annotations

import numpy as np
import pytest
import torch
import torch.nn.functional as F

import helion_mlir_utils as U
from tests.helpers import tensor, to_np

pytestmark = pytest.mark.gpu

RNG = np.random.default_rng(31)


def _matrix(rows: int, cols: int, pad: int, offset: int, device: torch.device) -> torch.Tensor:
    """An f32 [rows, cols] of row stride cols + pad, `offset` elements past a
    16-byte boundary, everything around it NaN."""
    pitch = cols + pad
    buf = torch.full((rows * pitch + offset + 64,), float("nan"), device=device)
    view = buf[offset:offset + rows * pitch].view(rows, pitch)[:, :cols]
    view.copy_(tensor(RNG.normal(0, 1, (rows, cols)).astype(np.float32), "f32", device))
    return view


def _check(got: np.ndarray, ref: np.ndarray, a: np.ndarray, b: np.ndarray) -> None:
    k = a.shape[-1]
    bound = 2 * k * 2.0 ** -24 * (np.abs(a).astype(np.float64) @ np.abs(b).astype(np.float64)) + 1e-6
    assert got.shape == ref.shape
    assert (np.abs(got.astype(np.float64) - ref) <= bound).all()


# Tiles of 32: one row, an edge, a full tile and one past it; K of 256 (one step
# a wave), one past, no multiple of 32, and the longest that few tiles take.
@pytest.mark.parametrize(("m", "n"), [(1, 1), (1, 333), (31, 33), (64, 64), (65, 127), (200, 1000)])
@pytest.mark.parametrize("k", [256, 257, 301, 1000])
@pytest.mark.parametrize(("trans_a", "trans_b"), [(False, False), (False, True), (True, False), (True, True)])
@pytest.mark.parametrize(("pad", "offset"), [(0, 0), (3, 1)])
def test_small_product(gpu_device, m: int, n: int, k: int, trans_a: bool, trans_b: bool, pad: int,
                       offset: int) -> None:
    a = _matrix(*((k, m) if trans_a else (m, k)), pad, offset, gpu_device)
    b = _matrix(*((n, k) if trans_b else (k, n)), pad, offset, gpu_device)
    an = to_np(a).T if trans_a else to_np(a)
    bn = to_np(b).T if trans_b else to_np(b)
    got = to_np(U.matmul(a, b, trans_a=trans_a, trans_b=trans_b))
    _check(got, an.astype(np.float64) @ bn.astype(np.float64), an, bn)


@pytest.mark.parametrize(("m", "n", "k"), [(33, 100, 300), (16, 2048, 2048)])
def test_epilogue_and_output_type(gpu_device, m: int, n: int, k: int) -> None:
    a, b = _matrix(m, k, 0, 0, gpu_device), _matrix(n, k, 0, 0, gpu_device)
    bias = tensor(RNG.normal(0, 1, n).astype(np.float32), "f32", gpu_device)
    an, bn = to_np(a), to_np(b).T
    ref = np.maximum(an.astype(np.float64) @ bn.astype(np.float64) + to_np(bias), 0)
    _check(to_np(U.matmul(a, b, trans_b=True, bias=bias, epilogue=F.relu)), ref, an, bn)
    out = to_np(U.matmul(a, b, trans_b=True, bias=bias, epilogue=F.relu, out_dtype=torch.bfloat16))
    # One rounding to bf16 (half an ulp, 2^-9) of an f32 sum within 1e-3.
    assert (np.abs(out - ref) <= 2.0 ** -8 * np.abs(ref) + 1e-3).all()


@pytest.mark.parametrize("shape", [(3, 40, 50, 515), (16, 32, 64, 256)])
def test_batches(gpu_device, shape: tuple[int, int, int, int]) -> None:
    s, m, n, k = shape
    a = tensor(RNG.normal(0, 1, (s, m, k)).astype(np.float32), "f32", gpu_device)
    b = tensor(RNG.normal(0, 1, (s, k, n)).astype(np.float32), "f32", gpu_device)
    an, bn = to_np(a), to_np(b)
    _check(to_np(U.bmm(a, b)), an.astype(np.float64) @ bn.astype(np.float64), an, bn)


def test_requested_splits_are_kept(gpu_device) -> None:
    a = tensor(RNG.normal(0, 1, (2, 64, 1024)).astype(np.float32), "f32", gpu_device)
    b = tensor(RNG.normal(0, 1, (2, 1024, 64)).astype(np.float32), "f32", gpu_device)
    an, bn = to_np(a), to_np(b)
    for splits in (1, 2, 8):
        _check(to_np(U.bmm(a, b, splits=splits)), an.astype(np.float64) @ bn.astype(np.float64), an, bn)
