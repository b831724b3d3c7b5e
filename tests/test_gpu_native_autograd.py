"""The native autograd functions (csrc/ca_torch.cpp) against the Python ones they
stand in for: equal bit for bit, and everything that is not the plain case
(transforms, duals, views, subclasses) still reaches the Python function."""
import threading

import pytest
import torch

pytestmark = pytest.mark.gpu


class _NoneExt:
    def __getattr__(self, name):
        return lambda *a: None


def _op_case(ca, dtype, D, T=150):
    g = torch.Generator().manual_seed(D)
    t = [torch.randn(2, 3, T, D, generator=g).to(dtype).cuda().requires_grad_() for _ in range(3)]
    r = (0.1 * torch.randn(3, generator=g)).cuda().requires_grad_()
    dy = torch.randn(2, 3, T, D, generator=g).to(dtype).cuda()

    def run():
        y = ca.continuum_attention(*t, r)
        return [y.detach(), *torch.autograd.grad(y, [*t, r], dy)]
    return run


def _rope_case(ca, dtype, theta):
    g = torch.Generator().manual_seed(1)
    x = torch.randn(2, 90, 3 * 4 * 32, generator=g).to(dtype).cuda().requires_grad_()
    r = (0.1 * torch.randn(4, generator=g)).cuda().requires_grad_()
    dy = torch.randn(2, 90, 4 * 32, generator=g).to(dtype).cuda()

    def run():
        y = ca.decoder.rope_continuum_attention(x, r, theta, 4)
        return [y.detach(), *torch.autograd.grad(y, [x, r], dy)]
    return run


def _norm_case(ca, res_dtype, use_sum):
    g = torch.Generator().manual_seed(2)
    norm = ca.decoder.RMSNorm(192).cuda()
    x = torch.randn(5, 7, 192, generator=g).cuda().requires_grad_()
    res = torch.randn(5, 7, 192, generator=g).to(res_dtype).cuda().requires_grad_()
    ds, dy = (torch.randn(5, 7, 192, generator=g).cuda() for _ in range(2))

    def run():
        with torch.autocast("cuda", dtype=torch.bfloat16, enabled=res_dtype == torch.bfloat16):
            y0 = norm(x)
            s, y = norm.add_and_norm(x, res)
        outs = [s, y, y0] if use_sum else [y, y0]
        go = [ds, dy.to(y.dtype), dy.to(y0.dtype)]
        return [o.detach() for o in outs] + list(
            torch.autograd.grad(outs, [x, res, norm.weight], go if use_sum else go[1:]))
    return run


def _weights_case(ca):
    g = torch.Generator().manual_seed(3)
    s = torch.randn(2, 3, 100, 100, generator=g).cuda().requires_grad_()
    gw = torch.randn(2, 3, 100, 100, generator=g).cuda()

    def run():
        w = ca.continuous_attention_weights(s)
        return [w.detach(), *torch.autograd.grad(w, s, gw)]
    return run


CASES = {
    "op_f32": lambda ca: _op_case(ca, torch.float32, 64),
    "op_bf16": lambda ca: _op_case(ca, torch.bfloat16, 64),
    "op_f16_padded": lambda ca: _op_case(ca, torch.float16, 40),
    "op_f32_padded": lambda ca: _op_case(ca, torch.float32, 20),
    "rope_bf16": lambda ca: _rope_case(ca, torch.bfloat16, 1e4),
    "rope_f32_none": lambda ca: _rope_case(ca, torch.float32, None),
    "norm_f32": lambda ca: _norm_case(ca, torch.float32, True),
    "norm_bf16_unused_sum": lambda ca: _norm_case(ca, torch.bfloat16, False),
    "weights": _weights_case,
}


@pytest.mark.parametrize("name", sorted(CASES))
def test_native_equals_python(gpu_ca, name, monkeypatch):
    run = CASES[name](gpu_ca)
    calls = []
    ext = gpu_ca.native.torch_ext()

    class _Spy:
        def __getattr__(self, f):
            def call(*a):
                r = getattr(ext, f)(*a)
                calls.append(r is not None)
                return r
            return call

    monkeypatch.setattr(gpu_ca.native, "torch_ext", _Spy)
    native = run()
    assert calls and all(calls)  # the native functions took every call
    packed = []
    with torch.autograd.graph.saved_tensors_hooks(lambda t: packed.append(1) or t.cpu(),
                                                  lambda t: t.cuda()):
        hooked = run()
    assert packed
    monkeypatch.setattr(gpu_ca.native, "torch_ext", _NoneExt)
    python = run()
    for a, b, c in zip(native, python, hooked):
        assert a.dtype == b.dtype and a.shape == b.shape
        assert torch.equal(a, b) and torch.equal(a, c)


def test_plain_case_only(gpu_ca):
    ca, ext = gpu_ca, gpu_ca.native.torch_ext()
    q = torch.randn(1, 2, 33, 32, device="cuda")
    g = torch.zeros(2, device="cuda")
    ref = ca.continuum_attention(q, q, q, g)
    view = torch.cat([q, q], -1)[..., :32]
    assert ext.op(view, q, q, g) is None and torch.equal(ca.continuum_attention(view, q, q, g), ref)
    off = torch.empty(q.numel() + 1, device="cuda")[1:].view_as(q).copy_(q)  # not 16-byte aligned
    assert ext.op(off, q, q, g) is None and torch.equal(ca.continuum_attention(off, q, q, g), ref)
    assert ext.op(q, q, q, g.double()) is None
    with pytest.raises(ValueError):
        ca.continuum_attention(q, q.half(), q, g)
    with pytest.raises(ValueError):
        ca.continuum_attention(q, q[:, :, :-1].contiguous(), q, g)
    with pytest.raises(ValueError):
        ca.continuum_attention(q, q, q, torch.zeros(3, device="cuda"))
    with pytest.raises(ValueError):
        ca.continuum_attention(q, q, q, g, 0)

    class Sub(torch.Tensor):
        pass

    assert ext.op(q.as_subclass(Sub), q, q, g) is None
    with pytest.raises(RuntimeError):  # a Function without setup_context under a transform
        torch.func.grad(lambda x: ca.continuum_attention(x, q, q, g).sum())(q)
    with pytest.raises(NotImplementedError), torch.autograd.forward_ad.dual_level():
        ca.continuum_attention(torch.autograd.forward_ad.make_dual(q, q), q, q, g)


def test_first_order_only_and_reuse(gpu_ca):
    q = torch.randn(1, 2, 20, 16, device="cuda", requires_grad=True)
    g = torch.zeros(2, device="cuda", requires_grad=True)
    y = gpu_ca.continuum_attention(q, q, q, g)
    a = torch.autograd.grad(y.sum(), [q, g], retain_graph=True)
    b = torch.autograd.grad(y.sum(), [q, g], retain_graph=True)
    assert all(torch.equal(s, t) for s, t in zip(a, b))
    with pytest.raises(RuntimeError, match="first-order"):
        torch.autograd.grad(y.sum(), q, create_graph=True)
    assert gpu_ca.continuum_attention(q.detach(), q.detach(), q.detach(), g.detach()).grad_fn is None
    with torch.no_grad():
        assert not gpu_ca.continuum_attention(q, q, q, g).requires_grad


def test_threads_and_streams(gpu_ca):
    """Each thread on a stream of its own: the same results as alone."""
    runs = [_op_case(gpu_ca, torch.float32, 64, T=300 + 10 * n) for n in range(3)]
    alone = [r() for r in runs]
    torch.cuda.synchronize()
    got = [None] * 3

    def work(n):
        s = torch.cuda.Stream()
        with torch.cuda.stream(s):
            for _ in range(3):
                got[n] = runs[n]()
        s.synchronize()

    threads = [threading.Thread(target=work, args=(n,)) for n in range(3)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for a, b in zip(alone, got):
        assert all(torch.equal(x, y) for x, y in zip(a, b))


@pytest.mark.parametrize("native", [True, False])
@pytest.mark.parametrize("name", ["op_f32", "op_f16_padded", "rope_bf16", "norm_f32",
                                  "norm_bf16_unused_sum", "weights"])
def test_saved_tensors_left_on_the_cpu_are_refused(gpu_ca, name, native, monkeypatch):
    """Saved-tensor hooks that do not bring the tensors back: an error, no kernel."""
    run = CASES[name](gpu_ca)
    if not native:
        monkeypatch.setattr(gpu_ca.native, "torch_ext", _NoneExt)
    for moved in (lambda n: True, lambda n: n == 1):  # every tensor, then the second alone
        count = []

        def unpack(t, moved=moved, count=count):
            count.append(1)
            return t.cpu() if moved(len(count) - 1) else t

        if name == "weights" and not moved(0):
            continue  # one saved tensor
        with torch.autograd.graph.saved_tensors_hooks(lambda t: t, unpack):
            with pytest.raises(RuntimeError, match="same|ROCm GPU|CUDA"):
                run()


@pytest.mark.parametrize("native", [True, False])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
def test_views_of_negated_values(gpu_ca, dtype, native, monkeypatch):
    """Tensors and gradients with the negative bit set (torch.conj and imag make
    them) are read as their values."""
    if not native:
        monkeypatch.setattr(gpu_ca.native, "torch_ext", _NoneExt)
    g = torch.Generator().manual_seed(4)
    q, k, v, dy = (torch.randn(1, 2, 70, 40, generator=g).to(dtype).cuda() for _ in range(4))
    gain = torch.zeros(2, device="cuda")
    norm = gpu_ca.decoder.RMSNorm(40).cuda()
    x, s = q[0].float(), torch.randn(2, 70, 70, generator=g).cuda()
    flip = torch._neg_view

    def run(neg):
        def arg(t):
            return (flip(-t) if neg else t.clone()).requires_grad_()

        out = []
        for f, args, grad in (
                (lambda *a: gpu_ca.continuum_attention(*a, gain), (q, k, v), dy),
                (lambda a: gpu_ca.decoder.rope_continuum_attention(a, gain, 1e4, 2),
                 (torch.cat([q[0, :, :, :32].reshape(1, 70, 64)] * 3, -1),),
                 dy[0, :, :, :32].reshape(1, 70, 64)),
                (norm, (x,), dy[0].float()),
                (lambda a, b: norm.add_and_norm(a, b)[1], (x, q[0]), dy[0].float()),
                (gpu_ca.continuous_attention_weights, (s,), s.flip(0))):
            leaves = [arg(t) for t in args]
            y = f(*leaves)
            out += [y.detach(), *torch.autograd.grad(y, leaves, flip(-grad) if neg else grad)]
        return out

    for a, b in zip(run(True), run(False)):
        assert torch.equal(a, b)
