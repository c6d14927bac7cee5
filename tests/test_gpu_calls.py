"""The native call path of nanoinfer_amd.quant: the same results as the Python path (reached
here by making the path decline), on side streams, and declined for everything but plain
calls, whose errors stay the Python path's."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _same(a, b):
    a, b = (a if isinstance(a, tuple) else (a,)), (b if isinstance(b, tuple) else (b,))
    assert len(a) == len(b)
    for x, y in zip(a, b):
        assert x.dtype == y.dtype and x.shape == y.shape and x.device == y.device and torch.equal(x, y)


@pytest.fixture
def declined(nq, monkeypatch):
    """Runs a call with the native path declining it."""
    names = ["linear", "gemm_w8a8", "act_quant", "act_quant_heads", "rmsnorm_quant", "add_rmsnorm_quant",
             "silu_mul_quant", "rope_qkv", "quantize"]

    def run(f):
        with monkeypatch.context() as mp:
            for n in names:
                mp.setattr(nq._calls, n, lambda *a: None)
            return f()
    return run


@pytest.mark.parametrize("dt", [torch.float32, torch.float16])
@pytest.mark.parametrize("m,n,k", [(1, 96, 256), (7, 33, 77), (40, 300, 1024), (0, 16, 64)])
def test_same_as_python_path(dev, nq, declined, dt, m, n, k):
    from nanoinfer_amd import model
    w = torch.randn(n, k, device=dev)
    x, b = torch.randn(m, k, device=dev).to(dt), torch.randn(n, device=dev)
    t8, t4 = nq.quantize_q8(w), nq.quantize_q4g(w, 32, torch.float16)
    r8, r4 = declined(lambda: nq.quantize_q8(w)), declined(lambda: nq.quantize_q4g(w, 32, torch.float16))
    _same((t8.q, t8.scale, t4.q, t4.scale), (r8.q, r8.scale, r4.q, r4.scale))
    assert (t8.out, t8.in_, t4.out, t4.in_, t4.group) == (n, k, n, k, 32)
    calls = [lambda o=o, f=f, t=t, bb=bb: f(x, t, bb, o) for o in (None, torch.float32, torch.float16) for bb in (None, b)
             for f, t in ((nq.linear_q8, t8), (nq.linear_q4g, t4), (nq.linear_w8a8, t8))]
    if m:
        xq, a_s = nq.act_quant(x)
        h, eps = torch.randn(k, device=dev), 1e-6
        gu = torch.randn(m, 2 * k, device=dev).to(dt)
        calls += [lambda: nq.act_quant(x), lambda: nq.gemm_w8a8(xq, a_s, t8, b, dt), lambda: nq.rmsnorm_quant(x, h, eps),
                  lambda: nq.add_rmsnorm_quant(x, x, h, eps), lambda: nq.silu_mul_quant(gu[:, :k], gu[:, k:])]
        _same(nq._calls.silu_mul_quant(gu, None), nq.silu_mul_quant(gu[:, :k].contiguous(), gu[:, k:].contiguous()))
        cos, sin = torch.randn(64, 32, device=dev), torch.randn(64, 32, device=dev)
        qkv = torch.randn(m, 8 * 32, device=dev).to(dt)
        heads = torch.randn(4, m, 32, device=dev).to(dt)
        calls += [lambda: model.rope_qkv(qkv, 4, 2, 32, cos, sin), lambda: nq.act_quant_heads(heads)]
    side = torch.cuda.Stream()
    for f in calls:
        ref = declined(f)
        _same(f(), ref)
        torch.cuda.synchronize()
        with torch.cuda.stream(side):
            y = f()
        side.synchronize()
        _same(y, ref)


def test_on_the_current_stream(dev, nq):
    """The launches queue on the current stream: behind a delay there, a copy into the input
    comes first. (Launched on any other stream they would read the old input.)"""
    from nanoinfer_amd import model
    m, k = 24, 512
    g = torch.Generator(device=dev).manual_seed(1)
    new = lambda *s: torch.randn(*s, generator=g, device=dev)
    t8, t4, h = nq.quantize_q8(new(300, k)), nq.quantize_q4g(new(300, k), 32), new(k)
    cos, sin = new(64, 64), new(64, 64)
    heads = lambda x: x.view(4, m, k // 4)
    calls = [lambda x: nq.linear_q8(x, t8), lambda x: nq.linear_q4g(x, t4), lambda x: nq.linear_w8a8(x, t8),
             lambda x: nq.gemm_w8a8(*nq.act_quant(x), t8), nq.act_quant, lambda x: nq.act_quant_heads(heads(x)),
             lambda x: nq.rmsnorm_quant(x, h, 1e-6), lambda x: nq.add_rmsnorm_quant(x, x, h, 1e-6),
             lambda x: nq.silu_mul_quant(x[:, :k // 2], x[:, k // 2:]), lambda x: nq._calls.silu_mul_quant(x, None),
             lambda x: model.rope_qkv(x, 4, 2, 64, cos, sin), lambda x: model.attention(*[x.view(8, m, 64)] * 3, 1),
             lambda x: (lambda t: (t.q, t.scale))(nq.quantize_q8(x)), lambda x: (lambda t: (t.q, t.scale))(nq.quantize_q4g(x, 32))]
    side = torch.cuda.Stream()
    for i, f in enumerate(calls):
        dt = torch.float16 if i in (2, 11) else torch.float32
        old, other = new(m, k).to(dt), new(m, k).to(dt)
        ref = f(other)
        x = old.clone()
        torch.cuda.synchronize()
        with torch.cuda.stream(side):
            torch.cuda._sleep(10_000_000)
            x.copy_(other)
            y = f(x)
        side.synchronize()
        _same(y, ref)


def test_data_pointer_that_throws(dev, nq):
    """A tensor without a data pointer: an error, from every call that asks for one."""
    x, t = torch.randn(4, 64, device=dev), nq.quantize_q8(torch.randn(16, 64, device=dev))
    torch._C._set_throw_on_mutable_data_ptr(x)
    for f in (lambda: nq.linear_q8(x, t), lambda: nq.linear_w8a8(x, t), lambda: nq.act_quant(x), lambda: nq.quantize_q8(x)):
        with pytest.raises(RuntimeError):
            f()


class Sub(torch.Tensor):
    pass


def test_declines_what_is_not_plain(dev, nq):
    x = torch.randn(4, 64, device=dev)
    t = nq.quantize_q8(torch.randn(16, 64, device=dev))
    c = lambda x, b=None, o=None, out=16, k=64, path=0: nq._calls.linear(0, x, t.q, t.scale, b, o, out, k, 0, path)
    assert c(x) is not None
    for bad in (x.t(), x[:, ::2], x.double(), x.cpu(), x[0], x[:, :32], x.as_subclass(Sub), None, 3):
        assert c(bad) is None
    assert c(x, b=torch.randn(15, device=dev)) is None and c(x, b=torch.randn(16, device=dev).half()) is None
    assert c(x, o=torch.float64) is None and c(x, o="f32") is None and c(x, path=9) is None and c(x, path="a") is None
    assert c(x, out=15) is None and c(x, out=-1) is None and c(x, k=65) is None
    with pytest.raises(ValueError):
        nq.linear_q8(x[:, :32], t)
    with pytest.raises(ValueError):
        nq.linear_q8(x, t, path=9)
    with pytest.raises(ValueError):
        nq.linear_q8(x, t, torch.randn(15, device=dev))
    _same(nq.linear_q8(torch.randn(64, 4, device=dev).copy_(x.t()).t(), t), nq.linear_q8(x, t))  # converted, as before
    with pytest.raises(TypeError):
        nq._calls.linear(1, 2)
