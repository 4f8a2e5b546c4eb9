"""LR reads with a token's row split over the waves of a workgroup: each source
slot count at its edges, 8- and 16-byte vectors, rows that end inside a wave,
heads of several waves, of a part of one and across two, one and several key
chunks and items per lane, the output norm and the bias, more tokens than
workgroups.  Against the oracle, with gpu_util's tolerances."""

import pytest
import torch

from test_gpu_parity import _lr_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("S", [2, 3, 4, 5, 6, 7, 8, 9, 10, 11, 12, 13, 14, 15, 16, 17, 20, 21, 24, 25, 28, 29, 32, 33, 40,
                               41, 48, 49, 56, 57, 64])
def test_split_read_source_slots(S):
    _lr_case(7000 + S, torch.bfloat16, 1, 3, 768, S, 64, 1, 0.125, True)


@pytest.mark.parametrize("S", [2, 6, 9, 14, 17, 25, 32])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
def test_split_read_wide_vectors(dtype, S):
    _lr_case(7100 + S, dtype, 1, 3, 1536, S, 32, 1, 0.125, True, normalize_output=True, bias=[0.1 * s for s in range(S)])


# D, R, H: whole rows of one head; heads of 1.5 waves, of 48 lanes, across waves; partial last waves; short and long key slices
_SHAPES = [(768, 32, 2), (768, 64, 4), (320, 8, 1), (640, 40, 5), (640, 128, 1), (2048, 128, 1), (1024, 64, 1), (192, 16, 1),
           (1344, 48, 3), (128, 128, 1)]


@pytest.mark.parametrize("D,R,Hh", _SHAPES)
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
def test_split_read_heads_and_rows(dtype, D, R, Hh):
    _lr_case(7200 + D + R, dtype, 2, 4, D, 11, R, Hh, 0.25, True, normalize_output=Hh == 1)
    _lr_case(7300 + D + R, dtype, 1, 2, D, 5, R, Hh, 0.25, False, bias=[0.3, -0.2, 0.7, 0.0, 0.4])


@pytest.mark.parametrize("norm", [False, True])
def test_split_read_walks_tokens(norm):
    _lr_case(7400, torch.bfloat16, 1, 4099, 192, 3, 16, 1, 0.25, True, normalize_output=norm)


@pytest.mark.parametrize("dtype,D,S,R,line", [(torch.float32, 1280, 17, 32, 512), (torch.float32, 1536, 3, 8, 512),
                                              (torch.bfloat16, 1536, 33, 32, 1024), (torch.float16, 1024, 41, 16, 2048)])
@pytest.mark.parametrize("norm", [False, True])
def test_split_read_forward_line(dtype, D, S, R, line, norm):
    """One token past the line the forward runs step by step (the backward stays split): results and gradients are those
    of the two parts, which take the split kernels, to the roundings of the order of fp32 sums: 16 of an fp32 ulp, or one
    step of the 16-bit type (2^-8, 2^-11 relative) in every element at worst."""
    import attnres_ops as ops

    g = torch.Generator(device="cuda").manual_seed(7500 + D)
    n, cut = line + 1, line // 2
    rn = lambda *s: torch.randn(s, generator=g, device="cuda").to(dtype)  # noqa: E731
    vals, keys, q, up = [rn(1, n, D) for _ in range(S)], [rn(1, n, R) for _ in range(S)], rn(1, R), rn(1, n, D)

    def run(a, b):
        vs, ks = ([t[:, a:b].contiguous().requires_grad_(True) for t in x] for x in (vals, keys))
        out = ops.lrid_attention_residual_read(vs, ks, q, 1, 0.25, True, normalize_output=norm)
        return [out.detach(), *torch.autograd.grad(out, [*vs, *ks], up[:, a:b].contiguous())]

    tol = {torch.float32: 2.0 ** -20, torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}[dtype]
    for whole, x, y in zip(run(0, n), run(0, cut), run(cut, n)):
        parts = torch.cat([x, y], 1).double()
        assert float((whole.double() - parts).norm() / parts.norm()) <= tol


def test_split_read_infinite_rows():
    """An infinity in a weighted source stays in its column; odd source counts pair the last row with zeros, not with itself."""
    import attnres_ops as ops
    from oracle import attnres_oracle as O

    g = torch.Generator().manual_seed(5)
    for S in (3, 9):
        vals = [torch.randn((1, 2, 768), generator=g).to(torch.bfloat16) for _ in range(S)]
        vals[-1][0, 0, 5] = float("inf")
        keys = [torch.randn((1, 2, 64), generator=g).to(torch.bfloat16) for _ in range(S)]
        q = torch.randn((1, 64), generator=g).to(torch.bfloat16)
        out = ops.lrid_attention_residual_read([v.cuda() for v in vals], [k.cuda() for k in keys], q.cuda(), 1, 0.125, True)
        ref = O.lrid_attention_residual_read_ref(vals, keys, q, 1, 0.125, True)
        assert torch.equal(torch.isinf(out.cpu()), torch.isinf(ref)) and not bool(torch.isnan(out).any())
