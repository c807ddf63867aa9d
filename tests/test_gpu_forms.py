"""Forward and dQ at the edges of their forms (row blocks x key groups): row
remainders of 32, 64 and 128, one row, key counts around multiples of the
groups' 64-key tiles (groups with fewer tiles or none), one to many
workgroups per head, causal grids that fold their tile order, and grids on
both sides of one and two rounds of the CUs. Every form that the rule picks, by
kernel, head-dim tile and mask, is among them (test_forms_rule.py checks that).
Against float32 autograd on the
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
    (1, 1, 1, 23, 29, False), (2, 8, 4, 1715, 2553, False), (2, 16, 4, 283, 270, False),
    (1, 1, 1, 23, 6080, False), (3, 4, 4, 1334, 741, True), (1, 1, 1, 1332, 1437, True),
    (3, 4, 2, 2518, 1099, True), (5, 9, 3, 1030, 1030, True), (2, 3, 3, 5873, 1254, True),
    (2, 3, 1, 5493, 1280, True), (1, 4, 2, 4197, 3140, True),
]


HEAD_DIMS = (32, 64, 80, 96, 128)


@pytest.mark.parametrize("d", HEAD_DIMS)
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


def _view(t, layout):
    """The same values with other strides: a model's [B, S, H, D] projection,
    or a slice of longer rows and a longer sequence."""
    if layout == "bshd":
        return t.transpose(1, 2).contiguous().transpose(1, 2)
    b, h, n, d = t.shape
    wide = torch.full((b, h, n + 5, d + 24), float("nan"), device=t.device, dtype=t.dtype)
    wide[:, :, :n, :d] = t
    return wide[:, :, :n, :d]


@pytest.mark.parametrize("d", [64, 80, 128])
@pytest.mark.parametrize("layout", ["bshd", "sliced"])
@pytest.mark.parametrize("shape", [
    (2, 16, 4, 449, 1537, False), (2, 8, 4, 1715, 2553, False), (2, 16, 16, 100, 3000, False),
    (1, 16, 8, 1029, 1029, False), (8, 8, 8, 512, 512, True), (1, 24, 8, 1990, 1990, True),
    (3, 4, 4, 1334, 741, True), (5, 9, 3, 1030, 1030, True),
], ids=str)
def test_forms_on_views_give_the_same_bits(shape, layout, d):
    b, hq, hkv, sq, sk, causal = shape
    dtype = torch.float16 if sq % 2 else torch.bfloat16
    q, k, v, do = (seeded(s, 700 + i, dtype=dtype) for i, s in enumerate(
        ((b, hq, sq, d), (b, hkv, sk, d), (b, hkv, sk, d), (b, hq, sq, d))))
    scale = 1 / math.sqrt(d)

    def run(view):
        out, lse = attention_forward(view(q), view(k), view(v), causal=causal, scale=scale)
        return out, lse, *attention_backward(view(q), view(k), view(v), view(out), lse, view(do),
                                             causal=causal, scale=scale)

    for name, e, a in zip(("O", "LSE", "dQ", "dK", "dV"), run(lambda t: t), run(lambda t: _view(t, layout))):
        assert torch.isfinite(a).all() and torch.equal(a, e), name
