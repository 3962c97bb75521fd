"""GEMMs of any number of rows against a packed B: the streaming kernel (up to
32 rows: one and two blocks of 16, K ranges shorter than its eight waves' steps)
and ragged 128 x 128 and 256 x 256 tiles, over every layout and panel width, N up to
and short of the padding. Against the CPU oracle; tolerance: one bf16
rounding of the result beside f32 sums (``bf16_gemm_atol``, rtol 1e-2).
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

RNG = np.random.default_rng(31)

LAYOUTS = {
    "vnni32": lambda bt: U.pack_b_vnni_t(bt, 32),
    "vnni64": lambda bt: U.pack_b_vnni_t(bt, 64),
    "vnni512": lambda bt: U.pack_b_vnni_t(bt, 512),
    "blocked": U.pack_b_blocked_t,
    "blocked_vnni": U.pack_b_blocked_vnni_t,
    "panels8": lambda bt: U.pack_b_panels(bt.t().contiguous(), 8),
    "panels128": lambda bt: U.pack_b_panels(bt.t().contiguous(), 128),
}


@pytest.mark.parametrize("m", [1, 16, 17, 32, 33, 127, 129, 300])
@pytest.mark.parametrize("layout", list(LAYOUTS))
def test_rows_against_packed_b(gpu_device, m: int, layout: str) -> None:
    for n, k in ((128, 256), (512, 320), (384, 64), (1152, 1088), (96, 288), (100, 512)):
        if layout.startswith("panels") and n % int(layout[6:]):
            continue
        a = tensor(RNG.normal(0, 1, (m, k)).astype(np.float32), "bf16", gpu_device)
        bt = tensor(RNG.normal(0, 1, (n, k)).astype(np.float32), "bf16", gpu_device)
        bias = tensor(RNG.normal(0, 1, n).astype(np.float32), "bf16", gpu_device)
        scale = tensor(RNG.normal(0, 1, n).astype(np.float32), "bf16", gpu_device)
        packed = LAYOUTS[layout](bt)
        an, bn = to_np(a), to_np(bt)
        atol = bf16_gemm_atol(k, an, bn)
        for act, kw, ref in ((U.identity_epilogue, {}, {}), (F.silu, {"scale": scale}, {"act": "silu", "scale": to_np(scale)}),
                             (torch.tanh, {}, {"act": "tanh"})):
            got = U.matmul_prepacked_b(a, packed, n, bias, act, **kw)
            assert got.shape == (m, n)
            assert_close(to_np(got), R.matmul(an, bn, False, True, to_np(bias), out="bf16", **ref), 1e-2, atol * 4)


@pytest.mark.parametrize("layout", ["vnni64", "panels128", "blocked"])
def test_big_ragged_tiles_against_packed_b(gpu_device, layout: str) -> None:
    # 3000 x 4096: 192 tiles of 256 x 256, M ragged; split K on 128 x 128 tiles.
    for m, n, k in ((3000, 4096, 512), (200, 1024, 4096)):
        a = tensor(RNG.normal(0, 1, (m, k)).astype(np.float32), "bf16", gpu_device)
        bt = tensor(RNG.normal(0, 1, (n, k)).astype(np.float32), "bf16", gpu_device)
        got = U.matmul_prepacked_b(a, LAYOUTS[layout](bt), n)
        an, bn = to_np(a), to_np(bt)
        assert_close(to_np(got), R.matmul(an, bn, False, True, out="bf16"), 1e-2, bf16_gemm_atol(k, an, bn))
