"""The C++ host side of the eager calls against the Python one: the same results
and gradients bit for bit over the forms both take (dtypes, layouts, options,
frozen inputs, odd sizes), the same answers where it stands aside, and autograd's
contracts (one backward only, saved-tensor hooks, in-place changes, transforms)."""

import contextlib

import pytest
import torch

import attnres_ops as ops

pytestmark = pytest.mark.gpu

BF = torch.bfloat16


@contextlib.contextmanager
def _python_route():
    saved, ops._NATIVE = ops._NATIVE, False
    try:
        yield
    finally:
        ops._NATIVE = saved


def _taken(monkeypatch_name, call):
    """Result of call() and whether the native entry answered it."""
    nat, seen = ops._native("forward", "backward"), []

    class Spy:
        def __getattr__(self, name):
            fn = getattr(nat, name)

            def wrapped(*a, **k):
                r = fn(*a, **k)
                seen.append((name, r is not None))
                return r

            return wrapped

    saved, ops._NATIVE = ops._NATIVE, Spy()
    try:
        return call(), (monkeypatch_name, True) in seen
    finally:
        ops._NATIVE = saved


def _flat(x):
    if isinstance(x, torch.Tensor):
        return [x]
    return [t for y in x for t in _flat(y)] if isinstance(x, (list, tuple)) else []


def _compare(name, make, call, native=True):
    """make(): named inputs (leaves); call(inputs): outputs.  Both routes, outputs and gradients."""
    res = []
    for route in (0, 1):
        torch.manual_seed(3)
        inp = make()
        leaves = [t for t in _flat(list(inp.values())) if t.requires_grad]
        if route == 0:
            out, took = _taken(name, lambda: call(inp))
            assert took == native
        else:
            with _python_route():
                out = call(inp)
        outs = [o for o in _flat(out)]
        diff = [o for o in outs if o.requires_grad]
        ups = [torch.randn_like(o) for o in diff]
        grads = torch.autograd.grad(diff, leaves, ups, allow_unused=True) if diff else []
        res.append((outs, grads))
    for a, b in zip(res[0][0], res[1][0]):
        assert a.shape == b.shape and a.dtype == b.dtype and torch.equal(a, b)
    assert len(res[0][1]) == len(res[1][1])
    for a, b in zip(res[0][1], res[1][1]):
        assert (a is None) == (b is None)
        if a is not None:
            assert a.shape == b.shape and a.dtype == b.dtype and torch.equal(a, b)


def _r(*shape, dtype=BF, grad=True, std=1.0):
    return (torch.randn(shape, device="cuda") * std).to(dtype).requires_grad_(grad)


_READS = {
    "lr": dict(B=2, T=5, D=256, R=32, H=2, N=3),
    "lr_wide": dict(B=1, T=7, D=768, R=64, H=1, N=5),
    "odd": dict(B=3, T=1, D=40, R=6, H=2, N=4),
    "one_token": dict(B=1, T=1, D=128, R=16, H=1, N=2),
    "many": dict(B=2, T=3, D=128, R=16, H=1, N=64),
}


@pytest.mark.parametrize("dtype", [torch.float32, BF, torch.float16])
@pytest.mark.parametrize("shape", list(_READS))
@pytest.mark.parametrize("norm,bias", [(False, None), (True, "list"), (True, "tensor")])
def test_reads(dtype, shape, norm, bias):
    c = _READS[shape]
    B, T, D, R, H, N = (c[k] for k in "BTDRHN")

    def make():
        b = [0.1 * s for s in range(N)] if bias == "list" else _r(N, dtype=torch.float32) if bias else None
        return dict(v=[_r(B, T, D, dtype=dtype) for _ in range(N)], k=[_r(B, T, R, dtype=dtype, grad=s % 2 == 0) for s in range(N)],
                    q=_r(H, R // H, dtype=dtype), qb=_r(D, dtype=dtype, std=0.1), qd=_r(B, T, H, R // H, dtype=dtype),
                    g=_r(B, T, H, dtype=dtype), g1=_r(H, dtype=dtype), sk=_r(N, R, dtype=dtype), b=b)

    kw = dict(normalize_output=norm)
    _compare("read", make, lambda i: ops.attention_residual_read(i["v"], i["qb"], True, source_logit_biases=i["b"], **kw))
    lr = ops.lrid_attention_residual_read
    _compare("read", make, lambda i: lr(i["v"], i["k"], i["q"], H, 0.25, True, source_logit_biases=i["b"], **kw))
    _compare("read", make, lambda i: lr(tuple(i["v"]), i["k"], i["qd"], H, 0.25, False, static_keys=i["sk"], **kw))
    gated = ops.lrid_attention_residual_read_gated
    _compare("read", make, lambda i: gated(i["v"], i["k"], i["q"], i["qd"], i["g"], H, 0.25, True, static_keys=i["sk"], **kw))
    _compare("read", make, lambda i: gated(i["v"], i["k"], None, i["qd"].reshape(B, T, R), i["g1"], H, 0.25, True, "linear", **kw))


@pytest.mark.parametrize("counts", [None, [1, 2, 3]])
def test_reads_views_and_no_grad(counts):
    def make():
        wide = _r(2, 4, 3 * 64 + 16)
        return dict(wide=wide, v=[wide[..., 64 * s:64 * (s + 1)] for s in range(3)], k=[wide[..., -16:]] * 3, q=_r(1, 16))

    call = lambda i: ops.lrid_attention_residual_read(i["v"], i["k"], i["q"], 1, 0.25, True, source_counts=counts)  # noqa: E731
    _compare("read", make, call)
    with torch.no_grad():
        i = make()
        a = call(i)
        with _python_route():
            assert torch.equal(a, call(i)) and not a.requires_grad


def test_calls_it_leaves_to_python():
    v = [_r(2, 4, 64) for _ in range(3)]
    k = [_r(2, 4, 16) for _ in range(3)]
    q = _r(1, 16)
    cases = [(torch.stack(v), k, q), (v, k, q.float()), ([v[0].float(), *v[1:]], k, q), (v, [t.float() for t in k], q),
             (v[:1], k[:1], q), ([t.transpose(0, 1).contiguous().transpose(0, 1) for t in v], k, q),
             ([v[0].expand(2, 4, 64), v[1][:, :1].expand(2, 4, 64), v[2]], k, q), ([t[:, :0] for t in v], [t[:, :0] for t in k], q)]
    for vs, ks, qq in cases:
        out, took = _taken("read", lambda: ops.lrid_attention_residual_read(vs, ks, qq, 1, 0.25, True))
        assert not took
        with _python_route():
            assert torch.equal(out, ops.lrid_attention_residual_read(vs, ks, qq, 1, 0.25, True))
    for bad in (dict(num_heads=3), dict(values=v[:2]), dict(query=q[:, :8])):
        a = dict(values=v, keys=k, query=q, num_heads=1, logit_scale=0.25, key_norm=True, **{})
        a.update(bad)
        with pytest.raises(RuntimeError) as e1:
            ops.lrid_attention_residual_read(**a)
        with _python_route(), pytest.raises(RuntimeError) as e2:
            ops.lrid_attention_residual_read(**a)
        assert str(e1.value) == str(e2.value)


@pytest.mark.parametrize("shape", [(2, 4, 8, 2), (2, 4, 1, 16), (2, 4, 16, 1), (4, 2, 2, 8), (1, 8, 2, 8)])
def test_a_per_token_query_of_another_shape_is_refused(shape):
    """[B, T, H, R/H] is [2, 4, 2, 8] here: as many elements in another order or for other heads are an error."""
    v, k = [_r(2, 4, 64) for _ in range(3)], [_r(2, 4, 16) for _ in range(3)]
    call = lambda: ops.lrid_attention_residual_read(v, k, _r(*shape), 2, 0.25, True)  # noqa: E731
    with pytest.raises(RuntimeError, match="per-token query must be") as e1:
        call()
    with _python_route(), pytest.raises(RuntimeError) as e2:
        call()
    assert str(e1.value) == str(e2.value)


def test_biases_and_queries_the_python_checks_judge():
    """A single source passes over its counts, sources may come from a generator, what was refused stays refused."""
    v, k = [_r(2, 4, 64) for _ in range(3)], [_r(2, 4, 16) for _ in range(3)]
    qb, q, qd = _r(64), _r(1, 16), _r(2, 4, 1, 16)
    base, lr, gated = ops.attention_residual_read, ops.lrid_attention_residual_read, ops.lrid_attention_residual_read_gated
    both = dict(source_counts=[1, 2, 3], source_logit_biases=[0.0, 0.1, 0.2])
    for call in (lambda: base(v[:1], qb, True, source_counts=[0]), lambda: lr(v[:1], k[:1], q, 1, 0.25, True, source_counts=[-1]),
                 lambda: gated(v[:1], k[:1], q, qd, None, 1, 0.25, True, source_counts=[0]),
                 lambda: base(v[:1], qb, True, source_counts=[1], source_logit_biases=[0.0]),
                 lambda: base((t for t in v), qb, True, source_counts=[1, 2, 3]),
                 lambda: lr((t for t in v), (t for t in k), q, 1, 0.25, True, source_logit_biases=[0.1, 0.2, 0.3])):
        got = call()
        with _python_route():
            assert torch.equal(got, call())
    for call in (lambda: gated(v, k, q, None, None, 1, 0.25, True), lambda: base(v, qb, True, source_counts=[1, 0, 2]),
                 lambda: lr(v, k, q, 1, 0.25, True, **both), lambda: base(v, qb, True, source_counts=[1, 2])):
        with pytest.raises((RuntimeError, AttributeError)) as e1:
            call()
        with _python_route(), pytest.raises((RuntimeError, AttributeError)) as e2:
            call()
        assert e1.type is e2.type and str(e1.value) == str(e2.value)


def _block(D=256, R=32, Q=3, S=3, T=5):
    return lambda: dict(v=[_r(2, T, D) for _ in range(S)], lg=[_r(Q, 2, T, dtype=torch.float32) for _ in range(S)],
                        y=[_r(2, T, D + R + 8) for _ in range(Q)], bank=_r(4, R), qs=_r(Q, D, std=0.1), pv=_r(2, T, D),
                        pk=_r(2, T, R), q=_r(D, std=0.1), inter=_r(2, T, D), lse=_r(2, T, dtype=torch.float32))


@pytest.mark.parametrize("D,R", [(256, 32), (768, 64)])
def test_block_calls(D, R):
    mk = _block(D, R)
    _compare("phase1_sources", mk, lambda i: ops.lrid_block_phase1(i["v"], i["lg"]))
    _compare("phase1_bank", mk, lambda i: ops.attention_residual_phase1(i["v"], i["qs"], True))
    for norm in (False, True):
        _compare("phase2", mk, lambda i: ops.attention_residual_phase2(i["pv"], i["q"], i["inter"], i["lse"], True,
                                                                       normalize_output=norm, logit_bias=0.7, partial_scale=0.5))
        for row, fn in ((None, ops.lrid_attention_residual_phase2), (2, ops.lrid_attention_residual_phase2_torch)):
            _compare("phase2", mk, lambda i: fn(i["pv"], i["pk"], i["bank"] if row is not None else i["bank"][1], i["inter"],
                                                i["lse"], 0.2, True, normalize_output=norm, query_row=row))
    _compare("block_accum", mk, lambda i: ops.lrid_block_accumulate(i["y"][0], None, None, D, R))
    _compare("block_accum", mk, lambda i: ops.lrid_block_accumulate(i["y"][0], i["pv"], i["pk"], D, R, complete=True,
                                                                    partial_scale=0.25))

    def chain(i):
        # the decoder's use: strided value gradients reach the earlier calls
        outs, lses = ops.lrid_block_phase1(i["v"], i["lg"])
        v = k = None
        hs = []
        for n in range(2):
            v, k, h = ops.lrid_block_accumulate_read(i["y"][n], v, k, i["bank"], outs[n + 1], lses[n + 1], D, R, 0.2,
                                                     lerp=True, normalize_output=True, logit_bias=0.1, partial_scale=0.5,
                                                     query_row=n)
            hs.append(h)
        return [*hs, *ops.lrid_block_accumulate(i["y"][2], v, k, D, R, complete=True, partial_scale=1 / 3)]

    _compare("accum_read", mk, chain)


def test_one_backward_only():
    v = [_r(1, 3, 64) for _ in range(2)]
    out = ops.attention_residual_read(v, _r(64), True)
    (g,) = torch.autograd.grad(out.float().square().sum(), [v[0]], create_graph=True)
    with pytest.raises(RuntimeError, match="once_differentiable"):
        g.float().sum().backward()


@pytest.mark.parametrize("route", [contextlib.nullcontext, _python_route])
def test_a_block_sources_gradient_outlives_the_others_alone(route):
    """Phase 1's value gradients are allocations of their own: one that is kept does not hold the others' memory."""
    i = _block(D=256, T=512)()
    with route():
        outs, _ = ops.lrid_block_phase1(i["v"], i["lg"])
        g = torch.autograd.grad(outs, i["v"], [torch.ones_like(o) for o in outs])
    assert len({t.untyped_storage().data_ptr() for t in g}) == len(g)


@pytest.mark.parametrize("name", ["read", "phase1", "bank", "phase2", "accum", "accum_read"])
def test_create_graph_under_a_constant_upstream_gradient(name):
    """create_graph with an upstream gradient that needs none: the gradients are constants of the next backward, on
    both routes (an incoming gradient that needs one makes them an error: test_one_backward_only)."""
    i = _block()()
    call = {"read": lambda: ops.attention_residual_read(i["v"], i["q"], True),
            "phase1": lambda: ops.lrid_block_phase1(i["v"], i["lg"])[0][1],
            "bank": lambda: ops.attention_residual_phase1(i["v"], i["qs"], True)[0],
            "phase2": lambda: ops.attention_residual_phase2(i["v"][0], i["q"], i["inter"], i["lse"], True),
            "accum": lambda: ops.lrid_block_accumulate(i["y"][0], i["pv"], i["pk"], 256, 32, complete=True)[0],
            "accum_read": lambda: ops.lrid_block_accumulate_read(i["y"][0], i["pv"], i["pk"], i["bank"], i["inter"],
                                                                 i["lse"], 256, 32, 0.2, query_row=1)[2]}[name]
    x = i["y"][0] if name.startswith("accum") else i["v"][0]

    def second():
        out = call()
        (g,) = torch.autograd.grad(out, [x], torch.ones_like(out), create_graph=True)
        assert not g.requires_grad
        return torch.autograd.grad((g.float() * x.float()).sum(), [x])[0]

    got = second()
    with _python_route():
        assert torch.equal(got, second())


def test_saved_tensor_hooks_and_in_place_changes():
    torch.manual_seed(1)
    v, q = [_r(1, 3, 64) for _ in range(3)], _r(64, std=0.2)
    ref = torch.autograd.grad(ops.attention_residual_read(v, q, True).float().sum(), [*v, q])
    with torch.autograd.graph.save_on_cpu():
        out = ops.attention_residual_read(v, q, True)
    for a, b in zip(torch.autograd.grad(out.float().sum(), [*v, q]), ref):
        assert torch.equal(a, b)
    w = [t * 1 for t in v]
    out = ops.attention_residual_read(w, q, True)
    w[1].add_(1)
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        out.float().sum().backward()


def _swapped(t):
    """The same values, the last two dimensions swapped in memory (or every second element of a row)."""
    if t.dim() < 2:
        out = t.new_empty((2 * t.numel(),))[::2].view(t.shape)
    else:
        out = t.new_empty((*t.shape[:-2], t.size(-1), t.size(-2))).transpose(-1, -2)
    return out.copy_(t)


def _shifted(t):
    """The same values, one element into a buffer."""
    return torch.cat([t.new_zeros(1), t.reshape(-1)])[1:].view(t.shape)


_HOOKED = {
    "base": lambda i: ops.attention_residual_read(i["v"], i["q"], True, normalize_output=True),
    "lr": lambda i: ops.lrid_attention_residual_read(i["v"], i["k"], i["qh"], 2, 0.25, True),
    "gated": lambda i: ops.lrid_attention_residual_read_gated(i["v"], i["k"], i["qh"], i["qd"], i["gate"], 2, 0.25, True,
                                                              static_keys=i["sk"]),
    "phase1": lambda i: ops.lrid_block_phase1(i["v"], i["lg"]),
    "bank": lambda i: ops.attention_residual_phase1(i["v"], i["qs"], True),
    "phase2": lambda i: ops.attention_residual_phase2(i["pv"], i["q"], i["inter"], i["lse"], True),
    "phase2_lr": lambda i: ops.lrid_attention_residual_phase2(i["pv"], i["pk"], i["bank"], i["inter"], i["lse"], 0.2, True,
                                                              query_row=1),
    "accum": lambda i: ops.lrid_block_accumulate(i["y"][0], i["pv"], i["pk"], 256, 32, complete=True, partial_scale=0.5),
    "accum_read": lambda i: ops.lrid_block_accumulate_read(i["y"][0], i["pv"], i["pk"], i["bank"], i["inter"], i["lse"], 256,
                                                           32, 0.2, query_row=1),
    "value_keys": lambda i: ops.lrid_value_key_projection(i["v"], i["bank_w"]),
}


@pytest.mark.parametrize("route", [contextlib.nullcontext, _python_route])
@pytest.mark.parametrize("name", list(_HOOKED))
@pytest.mark.parametrize("unpack", [_swapped, _shifted])
def test_saved_tensor_hooks_may_change_the_layout(unpack, name, route):
    torch.manual_seed(5)
    i = _block()()
    i.update(k=[_r(2, 5, 32) for _ in range(3)], qh=_r(2, 16), qd=_r(2, 5, 2, 16), gate=_r(2, 5, 2), sk=_r(3, 32),
             bank_w=_r(32, 256))
    leaves = [t for t in _flat(list(i.values())) if t.requires_grad]
    with route():
        def grads():
            outs = _flat(_HOOKED[name](i))
            torch.manual_seed(6)
            return torch.autograd.grad(outs, leaves, [torch.randn_like(o) for o in outs], allow_unused=True)

        want = grads()
        with torch.autograd.graph.saved_tensors_hooks(lambda t: t, unpack):
            got = grads()
    for a, b in zip(got, want):
        assert (a is None) == (b is None)
        if a is None:
            continue
        if unpack is _swapped:
            assert torch.equal(a, b)
        else:  # (kernels of another alignment may add in another order: an ulp of the largest element)
            assert (a.float() - b.float()).abs().max() <= 2.0 ** -7 * max(1.0, b.float().abs().max().item())


def test_transforms_and_modes_are_not_passed_by():
    v, q = [_r(1, 3, 64, grad=False) for _ in range(2)], _r(64, grad=False)
    with pytest.raises(RuntimeError, match="autograd.Function with functorch transforms"):
        torch.func.vmap(lambda a: ops.attention_residual_read([a, v[1]], q, True))(torch.stack([v[0], v[0]]))
    import torch.autograd.forward_ad as fwAD
    with fwAD.dual_level(), pytest.raises(NotImplementedError, match="forward mode AD"):
        d = fwAD.make_dual(v[0], torch.ones_like(v[0]))
        ops.attention_residual_read([d, v[1].requires_grad_()], q, True)

    class Sub(torch.Tensor):
        pass

    _, took = _taken("read", lambda: ops.attention_residual_read([v[0].as_subclass(Sub), v[0]], q, True))
    assert not took


def test_other_stream_and_thread():
    import threading

    v, q = [_r(4, 512, 1024) for _ in range(5)], _r(1024, std=0.05)
    ref = torch.autograd.grad(ops.attention_residual_read(v, q, True).float().sum(), [*v, q])
    torch.cuda.synchronize()
    got = {}

    def work(i):
        st = torch.cuda.Stream()
        with torch.cuda.stream(st):
            got[i] = torch.autograd.grad(ops.attention_residual_read(v, q, True).float().sum(), [*v, q])
        st.synchronize()

    ts = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    [t.start() for t in ts]
    [t.join() for t in ts]
    for i in range(4):
        for a, b in zip(got[i], ref):
            assert torch.equal(a, b)
