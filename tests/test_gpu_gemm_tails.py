"""bf16 GEMMs whose extents no tile divides, on the direct-to-LDS kernels: K
tails of every remainder, rows that keep 16-, 4- or 2-byte alignment, edges of
the 128 x 128 and 256 x 256 tiles, and batched products of transposed views.
Against the CPU oracle, with the memory around the operands filled with NaN:
a value read past a row's end that reached a product would show.

Tolerance: one bf16 rounding of the result beside f32 sums (``bf16_gemm_atol``,
rtol 1e-2), the suite's own for bf16 products.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch
import torch.nn.functional as F

import helion_mlir_utils as U
from oracle import restate as R
from tests.helpers import assert_close, bf16_gemm_atol, tensor, to_np

pytestmark = pytest.mark.gpu

RNG = np.random.default_rng(23)


def _matrix(rows: int, cols: int, pitch: int, offset: int, device: torch.device) -> torch.Tensor:
    """A bf16 [rows, cols] of row stride `pitch`, `offset` elements past a
    16-byte boundary, everything around it NaN."""
    buf = torch.full((rows * pitch + offset + 64,), float("nan"), dtype=torch.bfloat16, device=device)
    view = buf[offset:offset + rows * pitch].view(rows, pitch)[:, :cols]
    view.copy_(tensor(RNG.normal(0, 1, (rows, cols)).astype(np.float32), "bf16", device))
    return view


def _check(got: torch.Tensor, a: torch.Tensor, b: torch.Tensor, trans_a: bool, trans_b: bool, **kw) -> None:
    an, bn = to_np(a), to_np(b)
    k = an.shape[0] if trans_a else an.shape[1]
    ref = R.matmul(an, bn, trans_a, trans_b, out="f32" if got.dtype == torch.float32 else "bf16", **kw)
    assert_close(to_np(got), ref, 1e-2, bf16_gemm_atol(k, an, bn))


# Every remainder of a 64-deep stage that changes the path (a whole stage, one
# and all but one 8-element piece, pieces cut at even and odd elements), K of
# one to nine stages; 128 x 128 tiles.
@pytest.mark.parametrize("k", [2, 7, 8, 63, 64, 65, 66, 72, 100, 126, 127, 130, 191, 200, 322, 515, 570])
@pytest.mark.parametrize("trans_b", [False, True])
@pytest.mark.parametrize("pitch_pad", [0, 6, 8])
def test_k_tails(gpu_device, k: int, trans_b: bool, pitch_pad: int) -> None:
    m, n = 130, 144
    a = _matrix(m, k, k + pitch_pad, 0, gpu_device)
    b = _matrix(*((n, k) if trans_b else (k, n)), (k if trans_b else n) + pitch_pad, 0, gpu_device)
    for out in (None, torch.float32):
        _check(U.matmul(a, b, trans_b=trans_b, out_dtype=out), a, b, False, trans_b)


# Base pointers and N off every alignment, M and N at the tiles' edges.
@pytest.mark.parametrize(("m", "n"), [(1, 1), (65, 127), (128, 128), (129, 257), (33, 1003), (300, 258)])
@pytest.mark.parametrize("offset", [0, 1, 2, 4])
@pytest.mark.parametrize("trans_b", [False, True])
def test_unaligned_operands(gpu_device, m: int, n: int, offset: int, trans_b: bool) -> None:
    k = 202
    a = _matrix(m, k, k, offset, gpu_device)
    b = _matrix(*((n, k) if trans_b else (k, n)), k if trans_b else n, offset, gpu_device)
    bias = tensor(RNG.normal(0, 1, n).astype(np.float32), "bf16", gpu_device)
    got = U.matmul(a, b, trans_b=trans_b, bias=bias, epilogue=F.relu)
    _check(got, a, b, False, trans_b, bias=to_np(bias), act="relu")


# 256 x 256 tiles (fewer CUs than tiles): ragged everything, odd and even K,
# and A stored [K, M] transposed up front with a zero tail.
@pytest.mark.parametrize(("m", "n", "k"), [(4097, 4100, 72), (4096, 4096, 97), (4096, 4096, 100), (4090, 4098, 130)])
@pytest.mark.parametrize("trans_b", [False, True])
def test_big_tiles_with_tails(gpu_device, m: int, n: int, k: int, trans_b: bool) -> None:
    a = _matrix(m, k, k, 0, gpu_device)
    b = _matrix(*((n, k) if trans_b else (k, n)), k if trans_b else n, 0, gpu_device)
    _check(U.matmul(a, b, trans_b=trans_b), a, b, False, trans_b)


@pytest.mark.parametrize(("m", "n", "k"), [(513, 520, 514), (600, 777, 1001), (1024, 512, 2047)])
@pytest.mark.parametrize("trans_b", [False, True])
def test_transposed_a_with_tails(gpu_device, m: int, n: int, k: int, trans_b: bool) -> None:
    a = _matrix(k, m, m, 0, gpu_device)
    b = _matrix(*((n, k) if trans_b else (k, n)), k if trans_b else n, 0, gpu_device)
    _check(U.matmul(a, b, trans_a=True, trans_b=trans_b), a, b, True, trans_b)


# Other epilogues on a K tail (compiled in, and on the register-staged kernel
# where run-time compilation is off), programs, and split K with a tail in the
# last chunk.
@pytest.mark.parametrize("jit", ["1", "0"])
def test_epilogues_on_tails(gpu_device, monkeypatch, jit: str) -> None:
    monkeypatch.setenv("HMX_JIT", jit)
    for k in (100, 136):
        a, b = _matrix(200, k, k, 0, gpu_device), _matrix(k, 136, 136, 0, gpu_device)
        _check(U.matmul(a, b, epilogue=torch.tanh), a, b, False, False, act="tanh")
        program = lambda x: torch.relu(x) * 0.5 + 1.0  # noqa: E731
        _check(U.matmul(a, b, epilogue=program), a, b, False, False, act=program)


@pytest.mark.parametrize(("m", "n", "k"), [(512, 2048, 8184), (100, 130, 5000), (128, 128, 8200)])
@pytest.mark.parametrize("trans_b", [False, True])
def test_split_k_tails(gpu_device, m: int, n: int, k: int, trans_b: bool) -> None:
    a = _matrix(m, k, k, 0, gpu_device)
    b = _matrix(*((n, k) if trans_b else (k, n)), k if trans_b else n, 0, gpu_device)
    for splits in (None, 3):
        if splits is None:
            got = U.matmul(a, b, trans_b=trans_b)
        elif not trans_b:
            got = U.bmm(a[None], b[None], splits=splits)[0]
        else:
            got = U.bmm(a[None], b[None].transpose(1, 2), splits=splits)[0]
        _check(got, a, b, False, trans_b)


# Batched products: transposed views in place (any batch stride, an expanded
# batch), rows of every alignment, f32 too.
@pytest.mark.parametrize(("s", "m", "n", "k"), [(3, 40, 33, 64), (5, 130, 129, 80), (2, 1, 300, 66), (4, 70, 65, 35)])
@pytest.mark.parametrize("dtype", ["bf16", "f32"])
def test_bmm_transposed_views(gpu_device, s: int, m: int, n: int, k: int, dtype: str) -> None:
    def rand(*shape: int) -> torch.Tensor:
        return tensor(RNG.normal(0, 1, shape).astype(np.float32), dtype, gpu_device)

    a, keys = rand(s, m, k), rand(s, n, k)
    wide = rand(s, n + 3, k + 5)[:, 1:n + 1, 2:k + 2]  # strided rows and batches
    for b in (keys, wide, keys[:1].expand(s, n, k), keys.transpose(0, 1).contiguous().transpose(0, 1)):
        got, ref = to_np(U.bmm(a, b.transpose(1, 2))), to_np(U.bmm(a, b.transpose(1, 2).contiguous()))
        exact = np.einsum("smk,snk->smn", to_np(a).astype(np.float64), to_np(b).astype(np.float64))
        for r in (got, ref):
            if dtype == "f32":
                assert_close(r, exact, 1e-4, 1e-5 * np.sqrt(k))
            else:
                assert_close(r, exact, 1e-2, bf16_gemm_atol(k, to_np(a), to_np(b)))
