"""nq_attention_causal_f32 on the fp64 matrix cores, against the reference's arithmetic
in numpy (ops.cpp:206-270: double dot rounded to fp32, fp32 exp, double sums) at the
edges of its tiles of 16 queries and 16 keys, on both of its passes (scores kept in LDS
up to 2048 keys, recomputed past them) and with infinities and NaN."""
import numpy as np
import pytest
import torch

import model_ref as R

pytestmark = pytest.mark.gpu


def _run(q, k, v):
    from nanoinfer_amd import _lib
    h, s, d = q.shape
    D = lambda a: torch.from_numpy(np.ascontiguousarray(a, np.float32)).cuda()
    qd, kd, vd = D(q), D(k), D(v)
    out = torch.full((s, h * d), -7.0, device="cuda")
    _lib.check(_lib.load().nq_attention_causal_f32(qd.data_ptr(), kd.data_ptr(), vd.data_ptr(), h, k.shape[0], s, d,
                                                   out.data_ptr(), torch.cuda.current_stream().cuda_stream))
    return out.cpu().numpy().reshape(s, h, d).transpose(1, 0, 2)


def _inputs(h, kv, s, d, seed):
    r = np.random.default_rng(seed)
    n = lambda *a: r.normal(0, 1, a).astype(np.float32)
    return n(h, s, d) * 2, n(kv, s, d), n(kv, s, d)


# head size x length: one token, edges of one and several 16-row tiles, more tiles than
# the eight waves, the last length with saved scores and the first without.
@pytest.mark.parametrize("d", [32, 64, 96, 128])
@pytest.mark.parametrize("s", [1, 15, 16, 17, 130, 273])
def test_matches_reference(d, s):
    q, k, v = _inputs(4, 2, s, d, 3 * s + d)
    # Both sides round each score and each exp to fp32 from dots that differ by double
    # rounding only; a score may land on either neighbour, 2^-24 |score| of weight, and
    # expf differs from numpy's by an ulp: 8 * 2^-24 * max|v|, as the fixture test uses.
    ref = R.gqa_attention(q, k, v, 2)
    bound = 8 * 2.0 ** -24 * np.abs(v).max() * (1 + np.abs(q).max())
    assert np.abs(_run(q, k, v) - ref).max() <= bound


@pytest.mark.parametrize("d,s", [(32, 2048), (64, 2048), (32, 2049), (64, 2049), (96, 2063), (128, 2049)])
def test_long_rows(d, s):
    q, k, v = _inputs(1, 1, s, d, s)
    ref = R.gqa_attention(q, k, v, 1)
    bound = 8 * 2.0 ** -24 * np.abs(v).max() * (1 + np.abs(q).max())
    assert np.abs(_run(q, k, v) - ref).max() <= bound


@pytest.mark.parametrize("bad", [np.inf, -np.inf, np.nan])
@pytest.mark.parametrize("s,row", [(17, 16), (40, 35), (40, 3), (23, 22)])
def test_nonfinite_values_reach_only_later_queries(bad, s, row):
    q, k, v = _inputs(2, 1, s, 64, s + row)
    v[0, row, 5] = bad
    got = _run(q, k, v)
    clean = v.copy()
    clean[0, row, 5] = 0.0
    ref = _run(q, k, clean)
    assert np.array_equal(got[:, :row], ref[:, :row])
    cols = np.arange(64) != 5
    assert np.array_equal(got[:, row:, cols], ref[:, row:, cols])
    assert not np.isfinite(got[:, row:, 5]).any()


def test_nonfinite_scores():
    """A NaN score makes its query's row NaN and no other; keys past a query never count."""
    q, k, v = _inputs(1, 1, 33, 32, 5)
    q[0, 20, 1] = np.nan
    got = _run(q, k, v)
    q2 = q.copy()
    q2[0, 20] = 0
    ref = _run(q2, k, v)
    rows = np.arange(33) != 20
    assert np.array_equal(got[:, rows], ref[:, rows]) and np.isnan(got[0, 20]).all()
    k[0, 32] = np.inf  # the last key: only the last query sees it
    q2[0, 32] = -np.abs(q2[0, 32]) - 0.1  # a score of -inf: weight 0
    got = _run(q2, k, v)
    ref = R.gqa_attention(q2[:, :32], k[:, :32], v[:, :32], 1)
    assert np.isfinite(got).all() and np.abs(got[:, :32] - ref).max() <= 1e-5


def test_other_head_sizes_keep_the_general_kernel():
    q, k, v = _inputs(2, 1, 21, 40, 9)
    ref = R.gqa_attention(q, k, v, 2)
    assert np.abs(_run(q, k, v) - ref).max() <= 8 * 2.0 ** -24 * np.abs(v).max() * (1 + np.abs(q).max())
