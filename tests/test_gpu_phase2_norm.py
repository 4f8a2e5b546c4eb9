"""Base phase 2 with the fused output norm on the one-wave rows (and the widths and types that
stay on the step-by-step kernels), with and without key norm, learned bias and scale: against the
oracle with gpu_util's tolerances; 111 tokens leave part of the last workgroup idle."""

import pytest
import torch

from gpu_util import DEV, assert_close, gen, leaf, randn

import attnres_ops as ops
from oracle import attnres_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("D", [256, 512, 768, 1024, 640])
@pytest.mark.parametrize("key_norm,learned", [(True, False), (False, True), (True, True)])
def test_base_phase2_output_norm(dtype, D, key_norm, learned):
    g = gen(600 + D + key_norm + 2 * learned)
    B, T = 3, 37
    pv, it = randn(g, (B, T, D), dtype), randn(g, (B, T, D), dtype)
    q = randn(g, (D,), dtype, 1.5 / D ** 0.5)
    lse, up = randn(g, (B, T), torch.float32), randn(g, (B, T, D), dtype)
    bias = torch.tensor(0.3)

    def run(fn, dev, **kw):
        ins = [leaf(x, dev) for x in (pv, it, q, lse)]
        b = leaf(bias, dev) if learned else 0.3
        out = fn(ins[0], ins[2], ins[1], ins[3], key_norm, normalize_output=True, logit_bias=b, **kw)
        out.backward(up.to(dev))
        return [out, *[x.grad for x in ins], *([b.grad] if learned else [])]

    a, e = run(ops.attention_residual_phase2, DEV), run(O.attention_residual_phase2_ref, "cpu")
    for name, x, y in zip(("out", "dpartial", "dinter", "dq", "dlse", "dbias"), a, e):
        assert_close(x, y, dtype, name, reduced=name in ("dq", "dlse", "dbias"))
