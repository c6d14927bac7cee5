"""Causal fp16 attention (model.attention on heads of 64 and 128) against float64 on the
same fp16 inputs, at the edges of its tiles of 16 queries and 32 keys and of its four
waves, with infinities and NaN, and the calls that stay with torch."""
import math

import pytest
import torch

from test_spills import _spills


def _ref(q, k, v, n_rep):
    k, v = k.double().repeat_interleave(n_rep, 0), v.double().repeat_interleave(n_rep, 0)
    sc = torch.matmul(q.double(), k.transpose(1, 2).contiguous()) / math.sqrt(q.shape[2])
    s = q.shape[1]
    sc.masked_fill_(torch.ones(s, s, dtype=torch.bool, device=q.device).triu(1), -math.inf)
    return torch.matmul(torch.softmax(sc, -1), v)


def _inputs(h, kv, s, d, seed, dev):
    g = torch.Generator(device=dev).manual_seed(seed)
    n = lambda *a: torch.randn(*a, generator=g, device=dev).half()
    return n(h, s, d) * 2, n(kv, s, d), n(kv, s, d)


@pytest.mark.gpu
@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("s", [1, 2, 15, 16, 17, 31, 32, 33, 127, 129, 160, 515, 1024])
def test_matches_float64(dev, d, s):
    from nanoinfer_amd import model, quant
    q, k, v = _inputs(6, 2, s, d, s + d, dev)
    assert quant._calls.attention(q, k, v) is not None
    y, ref = model.attention(q, k, v, 3), _ref(q, k, v, 3)
    # the weights round to fp16 (2^-11 of each term, so of the weighted mean of |v|), as does
    # the result; fp32 scores of size |q||k| / sqrt(d) move a weight by 2^-22 of that size.
    lim = 2.0 ** -11 * _ref(q, k, v.abs(), 3) + 2.0 ** -11 * ref.abs() + 2.0 ** -15
    assert bool(((y.double() - ref).abs() <= lim).all())
    t = torch.nn.functional.scaled_dot_product_attention(q[None], k[None], v[None], is_causal=True, enable_gqa=True)[0]
    err = lambda a: float((a.double() - ref).norm() / ref.norm())
    assert err(y) <= 1.05 * err(t) + 1e-5  # no further off than the library call it replaces


@pytest.mark.gpu
@pytest.mark.parametrize("bad", [math.inf, -math.inf, math.nan])
@pytest.mark.parametrize("s,row", [(17, 16), (33, 20), (64, 40), (70, 3), (40, 39)])
def test_nonfinite_values_reach_only_later_queries(dev, bad, s, row):
    from nanoinfer_amd import model
    q, k, v = _inputs(4, 2, s, 128, s + row, dev)
    clean = model.attention(q, k, v, 2)
    v[0, row, 9] = bad
    y = model.attention(q, k, v, 2)
    cols = torch.arange(128, device=dev) != 9
    assert bool(torch.isfinite(y[:, :row]).all()) and bool(torch.isfinite(y[:, :, cols]).all())
    assert not bool(torch.isfinite(y[:2, row:, 9]).any()) and torch.equal(y[2:], clean[2:])
    assert float((y[:2, :row].float() - clean[:2, :row].float()).abs().max()) < 4e-3  # fp32 weights in that tile


@pytest.mark.gpu
def test_calls_that_stay_with_torch(dev):
    from nanoinfer_amd import model, quant
    q, k, v = _inputs(4, 2, 20, 64, 1, dev)
    c = quant._calls.attention
    assert c(q, k, v[:, :19]) is None and c(q, k.float(), v) is None and c(q.transpose(1, 2), k, v) is None
    assert c(q[:3].contiguous(), k, v) is None and c(q[..., :32].contiguous(), k[..., :32].contiguous(), v[..., :32].contiguous()) is None
    long = torch.zeros(2, 1025, 64, device=dev).half()
    assert c(long, long, long) is None and c(long[:, :1024].contiguous(), *[long[:, :1024].contiguous()] * 2) is not None
    for d, h, s, ours in ((128, 32, 768, True), (128, 32, 769, False), (128, 12, 2048, True), (128, 13, 2048, False),
                          (64, 24, 1024, True), (64, 25, 1024, False)):
        t = torch.zeros(h, s, d, device=dev).half()
        assert (c(t, t, t) is not None) == ours
        assert model.attention(t, t, t, 1).shape == t.shape
    qg = q.clone().requires_grad_()
    y = model.attention(qg, k, v, 2)
    y.float().sum().backward()
    assert qg.grad is not None and float((y.detach() - model.attention(q, k, v, 2)).abs().max()) < 4e-3


class _Seen(torch.overrides.TorchFunctionMode):
    def __init__(self):
        super().__init__()
        self.names = []

    def __torch_function__(self, func, types, args=(), kwargs=None):
        self.names.append(getattr(func, "__name__", ""))
        return func(*args, **(kwargs or {}))


@pytest.mark.gpu
@pytest.mark.parametrize("d", [64, 128])
def test_traced_and_steered_calls_stay_with_torch(dev, d):
    from nanoinfer_amd import model, quant
    from torch.nn.attention import SDPBackend, sdpa_kernel
    a, b = _inputs(4, 2, 33, d, 5, dev), _inputs(4, 2, 33, d, 6, dev)
    call = lambda q, k, v: model.attention(q, k, v, 2)
    traced = torch.jit.trace(call, a, check_trace=False)
    assert "scaled_dot_product_attention" in str(traced.graph)
    # both within the kernels' rounding of the other: 2^-11 of the values' size, a few times
    assert float((traced(*b).float() - call(*b).float()).abs().max()) < 4e-3
    with _Seen() as seen:
        call(*a)
    assert "scaled_dot_product_attention" in seen.names
    with sdpa_kernel(SDPBackend.MATH):
        assert quant._calls.attention(*a) is None
    with torch.autocast("cuda", dtype=torch.bfloat16):
        assert quant._calls.attention(*a) is None
    assert quant._calls.attention(*a) is not None


def test_compiles_as_one_graph():
    from nanoinfer_amd import model
    a = _inputs(4, 2, 20, 64, 7, "cpu")
    f = torch.compile(lambda q, k, v: model.attention(q, k, v, 2), backend="eager", fullgraph=True)
    assert torch.equal(f(*a), model.attention(*a, 2))


@pytest.mark.gpu
def test_inside_a_graph(dev):
    from nanoinfer_amd import model
    q, k, v = _inputs(4, 2, 90, 128, 2, dev)
    model.attention(q, k, v, 2)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        y = model.attention(q, k, v, 2)
    for i in range(3):
        q.copy_(_inputs(4, 2, 90, 128, i, dev)[0])
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, model.attention(q, k, v, 2))


def test_no_spills():
    assert not {k: v for k, v in _spills("nq_attention.hip").items() if v}
