"""Value-derived keys with their projection on the matrix cores: ranks 32 / 64 /
128, widths of one and of many steps and of partial column groups, token counts
around the 16-, 32- and 128-row tiles, several parts of the weight gradient's
tokens, row-strided and frozen inputs, and the forms that stay on the library
GEMM.  Against 64-bit closed forms: an output is at most a few bf16 roundings
(2^-9 each) off, relative to its norm."""

import pytest
import torch

import _attnres_hip as H
import attnres_ops as ops

pytestmark = pytest.mark.gpu

BF = torch.bfloat16


def _ref(vals, w, gk):
    v = [x.detach().double().requires_grad_(True) for x in vals]
    wd = w.detach().double().requires_grad_(True)
    keys = [(x * torch.rsqrt(x.square().mean(-1, keepdim=True) + torch.finfo(torch.float32).eps)) @ wd.t() for x in v]
    grads = torch.autograd.grad([k for k, g in zip(keys, gk) if g is not None], [*v, wd],
                                [g.double() for g in gk if g is not None], allow_unused=True)
    return keys, grads


def _close(a, e, name, bound=3 * 2.0 ** -9):
    a, e = a.detach(), e.detach()
    n = float(e.norm())
    assert float((a.double() - e).norm()) <= bound * n, (name, float((a.double() - e).norm()) / max(n, 1e-300))


def _check(N, B, T, D, R, fits=True, dtype=BF, drop=None, wide=0):
    torch.manual_seed(N * 1000 + T + D + R)
    base = [torch.randn((B, T, D + wide), device="cuda").to(dtype) for _ in range(N)]
    vals = [x[..., :D].requires_grad_(True) if not wide else x[..., :D].detach().requires_grad_(True) for x in base]
    w = (torch.randn((R, D), device="cuda") * D ** -0.5).to(dtype).requires_grad_(True)
    gk = [None if s == drop else torch.randn((B, T, R), device="cuda").to(dtype) for s in range(N)]
    assert H.value_keys_fits(H.ValueKey(vals), w.detach()) == fits
    keys = ops.lrid_value_key_projection(vals, w)
    grads = torch.autograd.grad([k for k, g in zip(keys, gk) if g is not None], [*vals, w],
                                [g for g in gk if g is not None], allow_unused=True)
    e_keys, e_grads = _ref(vals, w, gk)
    for s in range(N):
        _close(keys[s], e_keys[s], f"key{s}")
        if gk[s] is None:
            assert grads[s] is None or float(grads[s].abs().max()) == 0.0
        else:
            _close(grads[s], e_grads[s], f"dv{s}")
    _close(grads[-1], e_grads[-1], "dW")


@pytest.mark.parametrize("R", [32, 64, 128])
@pytest.mark.parametrize("D", [64, 192, 256, 320, 1024, 4096])
def test_widths_and_ranks(D, R):
    _check(3, 2, 37, D, R)


@pytest.mark.parametrize("n_tok", [1, 15, 16, 17, 31, 32, 33, 127, 128, 129, 511, 1025])
def test_token_counts(n_tok):
    _check(2, 1, n_tok, 256, 64)


@pytest.mark.parametrize("D,R,line", [(4096, 128, 16384), (3136, 128, 12544)])
def test_forward_line(D, R, line):
    """Rows up to the line take the norm and the library GEMM, one more the projection kernel; same keys either way, to
    the rounding of another order of fp32 sums (one bf16 step in every element at worst), with and without gradients."""
    torch.manual_seed(D + R)
    v = torch.randn((1, line + 1, D), device="cuda").to(BF)
    w = (torch.randn((R, D), device="cuda") * D ** -0.5).to(BF)
    with torch.no_grad():
        (more,), (up_to,) = (ops.lrid_value_key_projection([v[:, :n]], w) for n in (line + 1, line))
    _close(more[:, :line], up_to.double(), "keys", 2.0 ** -8)
    (k,) = ops.lrid_value_key_projection([v[:, :line].requires_grad_(True)], w)
    assert torch.equal(k.detach(), up_to)


def test_one_source_many_parts():
    _check(1, 1, 5000, 512, 128)


def test_sources_without_a_gradient_and_strided_rows():
    _check(4, 2, 40, 256, 32, drop=1)
    _check(3, 2, 40, 256, 32, wide=64)


@pytest.mark.parametrize("kw", [dict(dtype=torch.float16), dict(D=72), dict(R=48), dict(wide=4)])
def test_forms_of_the_library_gemm(kw):
    a = dict(N=2, B=1, T=20, D=128, R=32, fits=False)
    a.update(kw)
    _check(**a)


def test_frozen_inputs_rows_of_zeros_and_no_grad():
    torch.manual_seed(0)
    v = [torch.randn((1, 50, 256), device="cuda").to(BF) for _ in range(2)]
    v[0][:, 7] = 0
    w = (torch.randn((32, 256), device="cuda") * 0.06).to(BF)
    with torch.no_grad():
        ref = ops.lrid_value_key_projection(v, w)
    assert float(ref[0][:, 7].abs().max()) == 0.0
    a = v[0].clone().requires_grad_(True)
    keys = ops.lrid_value_key_projection([a, v[1]], w)
    assert all(torch.equal(x, y) for x, y in zip(keys, ref))
    (g,) = torch.autograd.grad(keys[0].float().sum() + keys[1].float().sum(), [a])
    assert bool(torch.isfinite(g).all())
    wl = w.clone().requires_grad_(True)
    keys = ops.lrid_value_key_projection(v, wl)
    (gw,) = torch.autograd.grad(keys[0].float().sum() + keys[1].float().sum(), [wl])
    _, e = _ref(v, w, [torch.ones_like(k) for k in keys])
    _close(gw, e[-1], "dW")
