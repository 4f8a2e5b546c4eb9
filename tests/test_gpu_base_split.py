"""Base reads with a token's row split over the waves of a workgroup: each source
slot count at its edges, 8- and 16-byte vectors, rows that end inside a wave or
a lane, the output norm, plain keys and the bias, more tokens than workgroups.
Against the oracle, with gpu_util's tolerances."""

import pytest
import torch

from test_gpu_parity import _base_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("S", [17, 20, 21, 24, 25, 28, 29, 32, 33, 40, 41, 48, 49, 56, 57, 64])
@pytest.mark.parametrize("D", [768, 1024])
def test_split_base_many_sources(S, D):
    _base_case(8000 + S, torch.bfloat16, 1, 3, D, S, True)


@pytest.mark.parametrize("S", [2, 3, 4, 5, 6, 7, 8, 9, 10, 11, 12, 13, 14, 15, 16])
def test_split_base_output_norm(S):
    _base_case(8100 + S, torch.bfloat16, 1, 3, 768, S, True, normalize_output=True)
    # plain keys: a query of 0.05 gives logits of order 0.05 * sqrt(1024) = 1.6.  At 0.5 they are of order 16, where an
    # fp16 logit has steps of 2^-6: one logit on a rounding tie then moves its weight by 1.6% and the query's gradient by
    # more than the 1e-3 mean bound (seen at S = 6, by the same 5.845e-3 from the step-by-step kernels)
    _base_case(8150 + S, torch.float16, 2, 2, 1024, S, False, normalize_output=True, bias=[0.1 * s for s in range(S)],
               qstd=0.05)


@pytest.mark.parametrize("D", [8, 64, 128, 320, 520, 640, 1536, 2040, 2048])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
def test_split_base_rows(dtype, D):
    # queries that give logits of order 1.6: at the helper's 0.5 they grow with sqrt(D) to about 60 at D = 1536, where fp32
    # sums carry 60 * 2^-24 * (a few) = 1e-5 into every weight, all of the fp32 bound (7.9e-6 of 0.73 seen)
    _base_case(8200 + D, dtype, 1, 4, D, 7, True, normalize_output=True, qstd=1.6 / D ** 0.5)
    _base_case(8300 + D, dtype, 1, 2, D, 18, False, bias=[0.05 * s for s in range(18)], qstd=1.6 / D ** 0.5)


@pytest.mark.parametrize("norm", [False, True])
def test_split_base_walks_tokens(norm):
    """Workgroups that walk several tokens give each token what a call of its own part gives it, bit for bit; the
    query's gradient, a sum over the tokens, to the rounding of its bf16 parts."""
    import attnres_ops as ops

    g = torch.Generator().manual_seed(8400)
    n, D, S = 8195, 640, 3
    vals = [torch.randn((1, n, D), generator=g).to(torch.bfloat16).cuda() for _ in range(S)]
    q = (torch.randn(D, generator=g) * 0.05).to(torch.bfloat16).cuda().requires_grad_(True)
    up = torch.randn((1, n, D), generator=g).to(torch.bfloat16).cuda()

    def run(a, b):
        vs = [v[:, a:b].contiguous().requires_grad_(True) for v in vals]
        out = ops.attention_residual_read(vs, q, True, normalize_output=norm)
        return [out, *torch.autograd.grad(out, [*vs, q], up[:, a:b].contiguous())]

    whole = run(0, n)
    parts = [run(a, min(a + 1000, n)) for a in range(0, n, 1000)]
    for i in range(S + 1):
        assert torch.equal(whole[i], torch.cat([x[i] for x in parts], 1)), i
    total = sum(x[-1].double() for x in parts)
    # nine parts rounded to bf16 (2^-9 each, relative) and the whole once
    assert float((whole[-1].double() - total).norm() / total.norm()) < 10 * 2.0 ** -9


@pytest.mark.parametrize("D,S,norm", [(640, 2, True), (1288, 2, False), (1288, 3, True)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_split_base_forward_line(dtype, D, S, norm):
    """2048 tokens of two or three such rows run the resident forward (the backward stays split): results and gradients are
    those of the halves, which take the split one, to the rounding of another order of fp32 sums, one step of the type in
    every element at worst."""
    import attnres_ops as ops

    g = torch.Generator(device="cuda").manual_seed(8500 + D)
    rn = lambda *s: torch.randn(s, generator=g, device="cuda").to(dtype)  # noqa: E731
    vals, q, up = [rn(1, 2048, D) for _ in range(S)], rn(D) * 0.03, rn(1, 2048, D)

    def run(a, b):
        vs = [v[:, a:b].contiguous().requires_grad_(True) for v in vals]
        out = ops.attention_residual_read(vs, q, True, normalize_output=norm)
        return [out.detach(), *torch.autograd.grad(out, vs, up[:, a:b].contiguous())]

    tol = 2.0 ** (-8 if dtype == torch.bfloat16 else -11)
    for whole, x, y in zip(run(0, 2048), run(0, 1024), run(1024, 2048)):
        parts = torch.cat([x, y], 1).double()
        assert float((whole.double() - parts).norm() / parts.norm()) <= tol


def test_split_base_infinite_rows():
    """An infinity in a source keeps out of the others: odd source counts pair the last row with zeros, not with itself."""
    import attnres_ops as ops
    from oracle import attnres_oracle as O

    g = torch.Generator().manual_seed(6)
    for S in (3, 19):
        vals = [torch.randn((1, 2, 640), generator=g).to(torch.bfloat16) for _ in range(S)]
        vals[-1][0, 0, 5] = float("inf")
        q = torch.zeros(640, dtype=torch.bfloat16)
        out = ops.attention_residual_read([v.cuda() for v in vals], q.cuda(), False)
        ref = O.attention_residual_read_ref(vals, q, False)
        assert torch.equal(torch.isnan(out.cpu()), torch.isnan(ref)) and torch.equal(torch.isinf(out.cpu()), torch.isinf(ref))
