"""Phase 1 from a query bank in one pass: every source and site slot count at
its edges, rows that fill a lane, a wave or eight waves and rows that do not,
more tokens than workgroups, and the shapes that stay on the composition.
Tolerances are gpu_util's (fp32 sums; 16-bit roundings where the eager op rounds)."""

import math

import pytest
import torch

from gpu_util import DEV, assert_close, gen, leaf, randn

import attnres_ops as ops
import _attnres_hip as H
from oracle import attnres_oracle as O

pytestmark = pytest.mark.gpu


def _check(dtype, S, Q, D, key_norm, n_tok, fits, lse_grad=True):
    g = gen(9000 + S * 31 + Q * 7 + D + n_tok)
    values = [randn(g, (1, n_tok, D), dtype) for _ in range(S)]
    queries = randn(g, (Q, D), torch.float32, 2.0 / math.sqrt(D))  # logits of order 2
    go = randn(g, (Q, 1, n_tok, D), dtype)
    glse = randn(g, (Q, 1, n_tok), torch.float32)
    vd = [leaf(x) for x in values]
    qd = leaf(queries)
    rows = [v.detach().view(n_tok, D) for v in vd]
    assert H.phase1_bank_fits(H.KeyedLogits(rows, qd.detach().to(dtype), key_norm)) == fits
    out, lse = ops.attention_residual_phase1(vd, qd, key_norm)
    vc = torch.stack(values).clone().requires_grad_(True)
    qc = queries.clone().requires_grad_(True)
    e_out, e_lse = O.attention_residual_phase1_ref(vc, qc, key_norm)
    if lse_grad:
        torch.autograd.backward([out, lse], [go.to(DEV), glse.to(DEV)])
        torch.autograd.backward([e_out, e_lse], [go, glse])
    else:
        out.backward(go.to(DEV))
        e_out.backward(go)
    assert_close(out, e_out, dtype, "out")
    assert_close(lse, e_lse, torch.float32 if dtype == torch.float32 else dtype, "lse", reduced=True)
    for s in range(S):
        assert_close(vd[s].grad, vc.grad[s], dtype, f"dv{s}")
    assert_close(qd.grad, qc.grad, dtype, "dqueries", reduced=True)
    with torch.no_grad():
        again, _ = ops.attention_residual_phase1([v.detach() for v in vd], qd.detach(), key_norm)
    assert torch.equal(again, out)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("S,Q,D,key_norm", [(1, 1, 256, True), (2, 1, 4, True), (3, 4, 252, True), (6, 5, 260, False),
                                            (7, 8, 640, True), (9, 12, 1024, True), (12, 9, 2048, True),
                                            (12, 12, 768, False)])
def test_query_bank_slots_and_rows(dtype, S, Q, D, key_norm):
    _check(dtype, S, Q, D, key_norm, 5, True)


@pytest.mark.parametrize("S,Q,D,key_norm,n_tok", [(2, 3, 64, True, 4099), (5, 2, 128, False, 1025), (4, 4, 256, True, 1)])
def test_query_bank_walks_tokens(S, Q, D, key_norm, n_tok):
    _check(torch.bfloat16, S, Q, D, key_norm, n_tok, True, lse_grad=n_tok != 1025)


@pytest.mark.parametrize("S,Q,D", [(13, 2, 256), (3, 13, 256), (3, 2, 254), (2, 2, 2052)])
def test_query_bank_shapes_of_the_composition(S, Q, D):
    _check(torch.bfloat16, S, Q, D, True, 3, False)


def test_query_bank_strided_sources_and_frozen_inputs():
    """Row views of wider tensors, a view off the vector alignment (composition), and only some inputs needing gradients."""
    g = gen(77)
    n, D, S, Q = 6, 256, 3, 2
    for off, fits in ((0, True), (64, True), (1, False)):
        wide = [randn(g, (1, n, D + 64 + off), torch.bfloat16).to(DEV) for _ in range(S)]
        vs = [w[..., off:off + D] for w in wide]
        v0 = vs[0].detach().requires_grad_(True)
        q = randn(g, (Q, D), torch.bfloat16, 0.1).to(DEV)
        rows = [v.detach()[0] for v in vs]
        assert H.phase1_bank_fits(H.KeyedLogits(rows, q, True)) == (fits and (D + 64 + off) % 4 == 0)
        out, lse = ops.attention_residual_phase1([v0, vs[1], vs[2]], q, True)
        (dv,) = torch.autograd.grad(out.float().sum() + lse.sum(), [v0])
        vc = torch.stack([v.detach().cpu() for v in vs]).requires_grad_(True)
        e_out, e_lse = O.attention_residual_phase1_ref(vc, q.cpu(), True)
        (e_dv,) = torch.autograd.grad(e_out.float().sum() + e_lse.float().sum(), [vc])
        assert_close(out, e_out, torch.bfloat16, "out")
        assert_close(dv, e_dv[0], torch.bfloat16, "dv")
