"""The tile GEMM (any k, alignment and group of whole chunks) through the public linears,
against float64 on the device at the edges of its tiles, slabs and split plans, and
against the wave-per-row kernels (NQ_PATH_GENERIC) on the same operands."""
import numpy as np
import pytest
import torch

from test_spills import _spills

F16, F32 = torch.float16, torch.float32
gpu = pytest.mark.gpu


def _codes(t, group):
    """Dequantized weights in float64 from the packed bytes."""
    if group == 0:
        return t.q.double() * t.scale.double()[:, None]
    nib = torch.stack([t.q & 15, t.q >> 4], 2).reshape(t.out, -1)[:, :t.in_].double() - 8
    return nib * t.scale.double().repeat_interleave(group, 1)[:, :t.in_]


def _make(nq, fmt, n, k, group, sdt, g):
    w = torch.randn(n, k, generator=g, device="cuda") * 0.02
    if fmt == "q8":
        return nq.quantize_q8(w), 0
    return (nq.quantize_q4g(w, group, sdt), group) if fmt == "q4g" else (nq.quantize_q4(w), max(1, k))


def _check(y, x, wd, b, k):
    """Any order of fp32 sums of exact products (three bf16 parts for fp32 x) is within
    3 k 2^-24 sum|x w|; scale, bias and the fp16 store round a few times more."""
    ref = x.double() @ wd.t().contiguous()
    lim = 3 * k * 2.0 ** -24 * (x.double().abs() @ wd.abs().t().contiguous())
    if b is not None:
        ref, lim = ref + b.double(), lim + 2.0 ** -22 * b.double().abs()
    lim = lim + 2.0 ** -21 * ref.abs()
    if y.dtype == F16:
        lim = lim + 2.0 ** -10 * ref.abs() + 2.0 ** -24
    assert y.shape == ref.shape
    assert bool(((y.double() - ref).abs() <= lim).all())
    if y.dtype == F32:  # the bound is loose by sqrt(k); test_errors_on_long_k has the tight one
        assert float((y.double() - ref).norm() / ref.norm()) < 2e-6


# one shape per tile and plan (whole and split K), k off every slab, odd n and m; then
# k below a chunk and a slab, exact slabs, one row of weights
PLANS = [(9, 65, 65), (9, 65, 2051), (400, 65, 2051), (700, 65, 1003), (33, 515, 2051), (130, 6001, 65),
         (257, 6001, 131), (257, 2003, 1003), (700, 515, 2051), (257, 4001, 1003), (520, 4001, 515), (777, 8960, 500),
         (1000, 4001, 325), (5, 1, 7), (9, 33, 31), (17, 130, 33), (64, 64, 320), (65, 129, 129), (16, 600, 1024)]

# the GEMVs of up to 8 rows: M buckets, pieces of 8 and 16 columns and their partial last
# one, K over 1, 2 and 4 waves, two and four weight rows per wave, ragged row counts
GEMVS = [(1, 1, 1), (1, 67, 15), (2, 130, 33), (3, 131, 1003), (8, 70, 1003), (5, 9, 8), (1, 515, 2051), (2, 70, 4099),
         (4, 66, 4099), (7, 67, 8191), (1, 8193, 259), (2, 8194, 131), (3, 8195, 67), (8, 8197, 131)]


@gpu
@pytest.mark.parametrize("xdt", [F32, F16])
@pytest.mark.parametrize("fmt,group", [("q8", 0), ("q4", 0), ("q4g", 32), ("q4g", 96), ("q4g", 128), ("q4g", 4096)])
def test_linear(dev, nq, xdt, fmt, group):
    g = torch.Generator(device=dev).manual_seed(group + len(fmt))
    for i, (m, n, k) in enumerate(PLANS):
        t, gr = _make(nq, fmt, n, k, group, F16 if i % 2 else F32, g)
        x = torch.randn(m, k, generator=g, device=dev).to(xdt)
        b = torch.randn(n, generator=g, device=dev) if i % 3 else None
        y = (nq.linear_q8 if fmt == "q8" else nq.linear_q4g)(x, t, b, F16 if i % 4 == 3 else F32)
        _check(y, x, _codes(t, gr), b, k)


@gpu
@pytest.mark.parametrize("m,n,k", PLANS + GEMVS + [(300, 200, 1040), (1122, 136, 5488), (16, 150, 1500), (520, 6001, 2051)])
def test_w8a8_exact(dev, nq, m, n, k):
    from nanoinfer_amd import _lib
    g = torch.Generator(device=dev).manual_seed(m + n + k)
    xq = torch.randint(-127, 128, (m, k), generator=g, device=dev, dtype=torch.int8)
    wq = torch.randint(-127, 128, (n, k), generator=g, device=dev, dtype=torch.int8)
    acc = nq.w8a8_acc_i32(xq, wq)
    assert torch.equal(acc.double(), xq.double() @ wq.double().t().contiguous())  # sums below 2^53
    t = nq.QTensor(wq, torch.rand(n, generator=g, device=dev) * 1e-3, n, k)
    a_s, b = torch.rand(m, generator=g, device=dev), torch.randn(n, generator=g, device=dev)
    for ydt in (F32, F16):
        got = nq.gemm_w8a8(xq, a_s, t, b, ydt)
        ref = nq.gemm_w8a8(xq, a_s, t, b, ydt, path=_lib.NQ_PATH_GENERIC)
        assert torch.equal(got, ref)


@gpu
@pytest.mark.parametrize("xdt", [F32, F16])
@pytest.mark.parametrize("fmt,group", [("q8", 0), ("q4", 0), ("q4g", 32), ("q4g", 96)])
def test_gemv(dev, nq, xdt, fmt, group):
    g = torch.Generator(device=dev).manual_seed(group + len(fmt))
    for i, (m, n, k) in enumerate(GEMVS):
        t, gr = _make(nq, fmt, n, k, group, F16 if i % 2 else F32, g)
        x = torch.randn(m, k, generator=g, device=dev).to(xdt)
        b = torch.randn(n, generator=g, device=dev) if i % 3 else None
        y = (nq.linear_q8 if fmt == "q8" else nq.linear_q4g)(x, t, b, F16 if i % 4 == 3 else F32)
        _check(y, x, _codes(t, gr), b, k)


# int8 on aligned rows of whole chunks, whose larger tiles add their sums in fp32
@gpu
@pytest.mark.parametrize("xdt", [F32, F16])
@pytest.mark.parametrize("m,n,k", [(1000, 4001, 1056), (1300, 5001, 1056)])
def test_q8_of_whole_chunks(dev, nq, xdt, m, n, k):
    g = torch.Generator(device=dev).manual_seed(n)
    t, _ = _make(nq, "q8", n, k, 0, F32, g)
    x, b = torch.randn(m, k, generator=g, device=dev).to(xdt), torch.randn(n, generator=g, device=dev)
    for ydt in (F32, F16):
        _check(nq.linear_q8(x, t, b, ydt), x, _codes(t, 0), b, k)


# Errors against 64 bits on long and odd K. The kernels before these summed K in 64 lanes
# and a tree; a result here rounds its sums over 256 columns (at most 8 additions that each
# hold j / 8 of the sum, (1 + ... + 8) / 8 = 4.5 roundings in quadrature; fp16 groups and
# int8 half as many), a plane (1), the end (1) and, for fp32 x, the three parts' MFMAs of a
# chunk (at most 3), each 2^-24 / sqrt(3) at most: sqrt(9.5) and sqrt(6.5) of these.
@gpu
@pytest.mark.parametrize("xdt", [F32, F16])
@pytest.mark.parametrize("fmt,group", [("q8", 0), ("q4", 0), ("q4g", 32), ("q4g", 64), ("q4g", 96), ("q4g", 256)])
def test_errors_on_long_k(dev, nq, xdt, fmt, group):
    g = torch.Generator(device=dev).manual_seed(group)
    lim = 2.0 ** -24 * ((9.5 if xdt == F32 else 6.5) / 3) ** 0.5
    for m, n, k in ((2, 8194, 301), (3, 8195, 149), (4, 200, 8955), (8, 2100, 1003), (12, 256, 1003), (130, 515, 8955),
                    (333, 4500, 8960 if fmt == "q4" else 9001), (600, 4001, 1003)):
        t, gr = _make(nq, fmt, n, k, group, F32, g)
        x = torch.randn(m, k, generator=g, device=dev).to(xdt)
        # odd rows: fp32 values whose three bf16 parts drop bits; fp16 subnormals
        x[1::2] *= 2.0 ** -116 if xdt == F32 else 2.0 ** -18
        ref = x.double() @ _codes(t, gr).t().contiguous()
        d = (nq.linear_q8 if fmt == "q8" else nq.linear_q4g)(x, t, None, F32).double() - ref
        for rows in (slice(0, None, 2), slice(1, None, 2)):
            assert float(d[rows].norm() / ref[rows].norm()) < lim, (m, n, k, rows)


@gpu
def test_nan_with_low_bits_only(dev, nq):
    """A NaN whose upper half reads as an infinity stays a NaN in every output of its row."""
    for m, k in ((3, 259), (40, 259), (300, 1003)):
        x = torch.randn(m, k, device=dev)
        x.view(torch.int32)[1, 7] = 0x7F800001
        for t, f in ((nq.quantize_q8(torch.randn(200, k, device=dev)), nq.linear_q8),
                     (nq.quantize_q4g(torch.randn(200, k, device=dev), 32), nq.linear_q4g)):
            y = f(x, t)
            assert bool(torch.isnan(y[1]).all()) and bool(torch.isfinite(y[0]).all()) and bool(torch.isfinite(y[2:]).all())


# fp32 rows: the errors have no common sign. The mean over 344064 outputs of errors of at
# most 3e-7 of the rms, were they independent, is within 3e-7 * 5 / 586; an eighth of
# 2^-24 leaves room for the products' own cut, and a sum cut once per chunk is over 3e-8.
@gpu
@pytest.mark.parametrize("fmt,group,k", [("q8", 0, 896), ("q8", 0, 4864), ("q4g", 32, 896), ("q4g", 32, 4864), ("q4g", 64, 896)])
def test_errors_have_no_mean(dev, nq, fmt, group, k):
    g = torch.Generator(device=dev).manual_seed(k)
    t, group = _make(nq, fmt, 896, k, group, F32, g)
    x = torch.randn(384, k, generator=g, device=dev)
    ref = x.double() @ _codes(t, group).t().contiguous()
    d = (nq.linear_q8 if fmt == "q8" else nq.linear_q4g)(x, t).double() - ref
    assert abs(float(d.mean() / ref.square().mean().sqrt())) < 2.0 ** -27


# the wave-per-row kernels stay behind an explicit path, over every type they take
@gpu
@pytest.mark.parametrize("ydt", [F32, F16])
@pytest.mark.parametrize("xdt", [F32, F16])
def test_explicit_generic_path(dev, nq, xdt, ydt):
    from nanoinfer_amd import _lib
    g = torch.Generator(device=dev).manual_seed(5)
    x, b = torch.randn(3, 203, generator=g, device=dev).to(xdt), torch.randn(65, generator=g, device=dev)
    for fmt, group, sdt in (("q8", 0, F32), ("q4g", 32, F32), ("q4g", 32, F16)):
        t, group = _make(nq, fmt, 65, 203, group, sdt, g)
        f = nq.linear_q8 if fmt == "q8" else nq.linear_q4g
        _check(f(x, t, b, out_dtype=ydt, path=_lib.NQ_PATH_GENERIC), x, _codes(t, group), b, 203)


@gpu
@pytest.mark.parametrize("xdt", [F32, F16])
def test_misaligned_rows_and_nonfinite_values(dev, nq, xdt):
    """Row starts off every alignment (views one element in), and infinities and NaN, which
    stay in their row and agree with the wave-per-row kernel."""
    from nanoinfer_amd import _lib
    g = torch.Generator(device=dev).manual_seed(3)
    for m, n, k in ((8, 33, 256), (8, 20, 259), (21, 70, 256), (40, 130, 259)):
        buf = torch.randn(m * k + 1, generator=g, device=dev).to(xdt)
        x = buf[1:].view(m, k)
        x[3, k - 1], x[5, 0], x[7, 40] = float("inf"), float("nan"), -float("inf")
        for t, f in ((nq.quantize_q8(torch.randn(n, k, generator=g, device=dev)), nq.linear_q8),
                     (nq.quantize_q4g(torch.randn(n, k, generator=g, device=dev), 32), nq.linear_q4g)):
            y, ref = f(x, t, None, F32), f(x, t, None, F32, path=_lib.NQ_PATH_GENERIC)
            assert torch.equal(torch.isnan(y), torch.isnan(ref)) and torch.equal(torch.isinf(y), torch.isinf(ref))
            rows = torch.ones(m, dtype=torch.bool, device=dev)
            rows[[3, 5, 7]] = False
            assert bool(torch.isfinite(y[rows]).all())
            assert float((y[rows] - ref[rows]).norm() / ref[rows].norm()) < 2e-6


# What stays with the kernels of 16 rows and 64-row split tiles: short K and fp32 x, few
# rows of x on a wide weight, fp16 x up to 64 rows (unsplit, split, and all output types).
KEPT = [(F32, 20, 300, 96), (F32, 40, 130, 160), (F32, 100, 130, 160), (F32, 20, 130, 2080), (F32, 12, 5000, 4128),
        (F32, 25, 4200, 160), (F16, 40, 300, 160), (F16, 100, 4200, 96), (F16, 24, 130, 2080), (F16, 40, 300, 2048),
        (F16, 24, 4200, 4128)]


@gpu
@pytest.mark.parametrize("xdt,m,n,k", KEPT)
@pytest.mark.parametrize("fmt,sdt", [("q8", F32), ("q4g", F32), ("q4g", F16)])
def test_neighbours_of_the_route(dev, nq, xdt, m, n, k, fmt, sdt):
    g = torch.Generator(device=dev).manual_seed(m + n)
    t, gr = _make(nq, fmt, n, k, 32, sdt, g)
    x = torch.randn(m, k, generator=g, device=dev).to(xdt)
    for ydt in (F32, F16):
        _check((nq.linear_q8 if fmt == "q8" else nq.linear_q4g)(x, t, None, ydt), x, _codes(t, gr), None, k)


def _call(lib, x, t, y, ws, nbytes, path):
    """nq_linear_q8_ex / nq_linear_q4g_ex on a workspace of the caller."""
    f = lambda d: 0 if d == F32 else 1
    tail = (None, y.data_ptr(), f(y.dtype), x.shape[0], t.out, t.in_, ws.data_ptr() if nbytes else None, nbytes, path,
            torch.cuda.current_stream().cuda_stream)
    if hasattr(t, "group"):
        return lib.nq_linear_q4g_ex(x.data_ptr(), f(x.dtype), t.q.data_ptr(), t.scale.data_ptr(), f(t.scale.dtype), t.group, *tail)
    return lib.nq_linear_q8_ex(x.data_ptr(), f(x.dtype), t.q.data_ptr(), t.scale.data_ptr(), *tail)


# The explicit MFMA path on the workspace that it requires splits K, as its planes there
# show: 64-row tiles of 64 and 128 columns, 16-row tiles of 17 to 32, 33 to 48 and more rows.
@gpu
@pytest.mark.parametrize("xdt", [F32, F16])
@pytest.mark.parametrize("m,n,k", [(40, 130, 2048), (100, 130, 2048), (24, 130, 4128), (24, 4200, 4128), (40, 130, 4128),
                                   (100, 130, 4128)])
def test_explicit_mfma_splits_k(dev, nq, xdt, m, n, k):
    from nanoinfer_amd import _lib
    lib, g = _lib.load(), torch.Generator(device=dev).manual_seed(m + n + k)
    x = torch.randn(m, k, generator=g, device=dev).to(xdt)
    need = lib.nq_linear_wq_workspace_size(m, n, k)
    assert need > 0
    for fmt, group, sdt in (("q8", 0, F32), ("q4g", 32, F32), ("q4g", 32, F16), ("q4g", 64, F32), ("q4g", 64, F16), ("q4g", 128, F32)):
        t, gr = _make(nq, fmt, n, k, group, sdt, g)
        for ydt in (F32, F16):
            ws = torch.full((need,), 255, dtype=torch.uint8, device=dev)
            y = torch.empty(m, n, dtype=ydt, device=dev)
            _lib.check(_call(lib, x, t, y, ws, need, _lib.NQ_PATH_MFMA))
            _check(y, x, _codes(t, gr), None, k)
            assert bool((ws != 255).any()), (fmt, group, sdt, ydt)


@gpu
def test_less_workspace_splits_less(dev, nq):
    """The plain entries (no workspace) and a workspace below the preferred size give the
    same result up to the order of the sums."""
    from nanoinfer_amd import _lib
    lib, m, n, k = _lib.load(), 70, 600, 2019
    best = lib.nq_linear_wq_workspace_preferred(m, n, k)
    assert best >= 2 * m * n * 4 and lib.nq_linear_wq_workspace_size(m, n, k) == 0
    t = nq.quantize_q8(torch.randn(n, k, device=dev))
    x = torch.randn(m, k, device=dev)
    full = nq.linear_q8(x, t)
    ws = torch.empty(best, dtype=torch.uint8, device=dev)
    y = torch.empty_like(full)
    for nbytes in (0, m * n * 4, best // 2):
        y.fill_(-1)
        _lib.check(lib.nq_linear_q8_ws(x.data_ptr(), 0, t.q.data_ptr(), t.scale.data_ptr(), None, y.data_ptr(), 0, m, n, k,
                                       ws.data_ptr() if nbytes else None, nbytes, torch.cuda.current_stream().cuda_stream))
        assert float((y - full).norm() / full.norm()) < 1e-6


@gpu
@pytest.mark.parametrize("m,n,k", [(32, 128, 1024), (100, 128, 1536), (48, 128, 1024)])
def test_required_workspace_keeps_the_kernel(dev, nq, m, n, k):
    """With the required workspace only, of which the tile GEMM would need far more, fp32 rows
    stay on the kernel whose planes that size holds (the explicit MFMA path, bit for bit)."""
    from nanoinfer_amd import _lib
    lib = _lib.load()
    need, best = lib.nq_linear_wq_workspace_size(m, n, k), lib.nq_linear_wq_workspace_preferred(m, n, k)
    assert 0 < need < best
    ws = torch.empty(best, dtype=torch.uint8, device=dev)
    x = torch.randn(m, k, device=dev)
    for t, gr in (_make(nq, "q8", n, k, 0, F32, None), _make(nq, "q4g", n, k, 32, F32, None)):
        y, ref = torch.empty(m, n, device=dev), torch.empty(m, n, device=dev)
        _lib.check(_call(lib, x, t, ref, ws, need, _lib.NQ_PATH_MFMA))
        _lib.check(_call(lib, x, t, y, ws, need, _lib.NQ_PATH_AUTO))
        assert torch.equal(y, ref)
        _lib.check(_call(lib, x, t, y, ws, best, _lib.NQ_PATH_AUTO))
        _check(y, x, _codes(t, gr), None, k)


# Calls that the tile GEMM or the GEMVs of any k are slower for: bit for bit the kernels of
# the explicit paths.
@gpu
@pytest.mark.parametrize("xdt,m,n,k,fmt,group", [
    (F32, 39, 3648, 512, "q8", 0), (F32, 20, 7424, 1664, "q4g", 32), (F32, 24, 512, 4096, "q8", 0), (F32, 46, 256, 7168, "q4g", 64),
    (F32, 20, 512, 256, "q4", 0), (F16, 19, 320, 512, "q4", 0), (F16, 43, 3392, 1024, "q4g", 32), (F16, 333, 1536, 8960, "q4g", 64)])
def test_kept_on_mfma(dev, nq, xdt, m, n, k, fmt, group):
    from nanoinfer_amd import _lib
    t, gr = _make(nq, fmt, n, k, group, F32, None)
    x = torch.randn(m, k, device=dev).to(xdt)
    f = nq.linear_q8 if fmt == "q8" else nq.linear_q4g
    assert torch.equal(f(x, t), f(x, t, path=_lib.NQ_PATH_MFMA))


@gpu
@pytest.mark.parametrize("xdt", [F32, F16])
@pytest.mark.parametrize("m,n,k", [(1, 2358, 65), (2, 6462, 87), (2, 60, 159), (1, 60, 255), (5, 426, 51), (8, 90, 111)])
def test_kept_on_elements(dev, nq, xdt, m, n, k):
    from nanoinfer_amd import _lib
    t, _ = _make(nq, "q8", n, k, 0, F32, None)
    x = torch.randn(m, k, device=dev).to(xdt)
    assert torch.equal(nq.linear_q8(x, t), nq.linear_q8(x, t, path=_lib.NQ_PATH_GENERIC))


def test_workspace_sizes_of_short_k():
    """Shapes below one 32-column chunk: no workspace is required (a division by the
    number of chunks once stood here)."""
    from nanoinfer_amd import _lib
    lib = _lib.load()
    for m in (1, 9, 64, 300):
        for k in (1, 7, 31):
            assert lib.nq_linear_wq_workspace_size(m, 100, k) == 0
            assert lib.nq_linear_wq_workspace_preferred(m, 100, k) % 256 == 0


def test_no_spills():
    for src in ("nq_tile_gemm.hip", "nq_gemv_any.hip"):
        assert not {k: v for k, v in _spills(src).items() if v}
