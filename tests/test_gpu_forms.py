"""Forward and dQ at the edges of their forms (row blocks x key groups): row
remainders of 32, 64 and 128, one row, key counts around multiples of the
groups' 64-key tiles (groups with fewer tiles or none), one to many
workgroups per head, causal grids that fold their tile order, and grids on
both sides of one and two rounds of the CUs. Against float32 autograd on the
same inputs, at the bars of the other forward and backward tests (dK and dV, which
have no forms, in fp16 only)."""
import math

import pytest
import torch

from kotflash_amd.kernels.hip_backward import attention_backward
from kotflash_amd.kernels.hip_forward import attention_forward
from tests.gpu_helpers import BWD_TOL, BWD_TOL_BF16_SHORT, FWD_TOL, assert_close, reference_fp32, seeded

pytestmark = pytest.mark.gpu

SHAPES = [  # b, hq, hkv, sq, sk, causal
    (1, 2, 2, 1, 129, False), (2, 16, 16, 100, 3000, False), (1, 16, 8, 448, 1500, False),
    (2, 16, 4, 449, 1537, False), (4, 8, 8, 300, 1500, False), (1, 16, 16, 1024, 1024, False),
    (3, 4, 4, 65, 191, False), (8, 8, 8, 512, 512, True), (1, 16, 8, 2048, 2048, True),
    (1, 24, 8, 1990, 1990, True), (2, 8, 2, 1025, 700, True), (1, 32, 8, 1777, 1777, True),
    (16, 8, 8, 200, 90, True), (2, 4, 1, 97, 2000, True),
]


@pytest.mark.parametrize("d", [32, 64, 80, 96, 128])
@pytest.mark.parametrize("shape", SHAPES, ids=str)
def test_forms_against_fp32(shape, d):
    b, hq, hkv, sq, sk, causal = shape
    dtype = torch.float16 if (sq + d // 16) % 2 else torch.bfloat16
    q, k, v, do = (seeded(s, 600 + i, dtype=dtype) for i, s in enumerate(
        ((b, hq, sq, d), (b, hkv, sk, d), (b, hkv, sk, d), (b, hq, sq, d))))
    scale = 1 / math.sqrt(d)
    out, lse = attention_forward(q, k, v, causal=causal, scale=scale)
    dq, dk, dv = attention_backward(q, k, v, out, lse, do, causal=causal, scale=scale)
    eo, el, (eq, ek, ev) = reference_fp32(q, k, v, causal=causal, with_grad_out=do)
    assert_close(out, eo, **FWD_TOL[dtype], what="O")
    assert_close(lse, el, **FWD_TOL[dtype], what="LSE")
    tol = BWD_TOL[dtype] if dtype == torch.float16 else BWD_TOL_BF16_SHORT
    assert_close(dq, eq, **tol, what="dQ")
    if dtype == torch.float16:
        assert_close(dk, ek, **tol, what="dK")
        assert_close(dv, ev, **tol, what="dV")
