"""dK/dV at the edges of its share plans: shares of whole tile rows (with and
without room to spare), rows cut into many shares (the fixup's batches of four
and their remainders) or into few (whose shares are shorter), fewer shares than
CUs, a single unit, and keys that no query sees. Against float32 autograd at the
backward's fp16 bar; dK/dV sum up to 8 heads of a group, so the outputs are
scaled to a few units at most."""
import math

import pytest
import torch

from kotflash_amd.kernels.hip_backward import attention_backward
from kotflash_amd.kernels.hip_forward import attention_forward
from tests.gpu_helpers import BWD_TOL, assert_close, reference_fp32, seeded

pytestmark = pytest.mark.gpu
F16 = torch.float16


@pytest.mark.parametrize("d", [64, 80, 128])
@pytest.mark.parametrize("shape", [
    (4, 12, 12, 1000, 1000, True), (4, 16, 16, 512, 512, True), (3, 8, 8, 640, 640, False),
    (1, 8, 1, 700, 700, False), (1, 8, 1, 700, 700, True), (2, 8, 2, 1024, 1024, True),
    (1, 1, 1, 1, 1, True), (1, 1, 1, 64, 129, False), (2, 4, 1, 200, 900, True),
    (1, 32, 4, 500, 500, True), (8, 12, 12, 1024, 1024, True),
    (3, 16, 8, 533, 533, True), (1, 16, 4, 433, 433, True), (3, 8, 1, 88, 2355, False),
], ids=str)
def test_dkdv_share_plans(shape, d):
    b, hq, hkv, sq, sk, causal = shape
    q, k, v, do = (seeded(s, 800 + i, dtype=F16) * 0.5 for i, s in enumerate(
        ((b, hq, sq, d), (b, hkv, sk, d), (b, hkv, sk, d), (b, hq, sq, d))))
    scale = 1 / math.sqrt(d)
    out, lse = attention_forward(q, k, v, causal=causal, scale=scale)
    got = attention_backward(q, k, v, out, lse, do, causal=causal, scale=scale)
    again = attention_backward(q, k, v, out, lse, do, causal=causal, scale=scale)
    _, _, exact = reference_fp32(q, k, v, causal=causal, with_grad_out=do)
    for name, g, a, e in zip(("dQ", "dK", "dV"), got, again, exact):
        assert_close(g, e, **BWD_TOL[F16], what=name)
        assert torch.equal(g, a), name
