"""QJL scores, weighted values and softmax at the edges of their tiles (16
queries and 64, 32 keys, chunks of 256 values, rows kept in registers up to
16,384 columns) against the oracle and float64 numpy.

Tolerances: scores as the oracle test of the C5 size, 1e-5 of |q| |k|;
weighted values 1e-5 of sum |w v|; softmax 1e-6 of its row's largest value
(an exponential's few ulps and an f32 sum of up to 20,000 terms)."""
import numpy as np
import pytest

from oracle import oracle as orc

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


@pytest.fixture(scope="module")
def tq():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import turboquant_amd
    return turboquant_amd


def _dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


@pytest.mark.parametrize("dim,tb,nk,nq", [(128, 3, 1, 1), (128, 4, 31, 15), (64, 3, 33, 17), (32, 4, 100, 65),
                                          (64, 4, 64, 64), (32, 3, 65, 16)])
def test_scores_at_tile_edges(tq, dim, tb, nk, nq):
    keys, qs = orc.lcg_normal_vecs(nk, dim, nk), orc.lcg_normal_vecs(7 + nq, dim, nq)
    keys[-1] *= 100.0
    qs[0] *= 1e-6
    recs = orc.qjl_quantize_batch(tb, dim, 42, 5, keys)
    ref = orc.qjl_scores(tb - 1, dim, 42, 5, qs, *recs)
    ctx = tq.qjl_query_context(_dev(qs), 42, 5)
    dev = [_dev(r.view(np.int16) if r.dtype == np.uint16 else r) for r in recs]
    got = tq.qjl_scores(ctx, *dev, tb - 1, 42).cpu().numpy()
    natural = np.linalg.norm(qs, axis=1)[:, None] * np.linalg.norm(keys, axis=1)[None, :]
    assert (np.abs(got - ref) / natural).max() <= 1e-5


@pytest.mark.parametrize("dim,tb", [(128, 3), (64, 4), (32, 3)])
def test_scores_of_tiny_queries(tq, dim, tb):
    """A context times 2^-122 gives the scores times 2^-122: its elements are rounded to 2^-149, 2^-27 of them, and
    each score once more (2^-24): 1e-6 of the row's root mean square.  Rows on a clamped scale are off by 3e-5."""
    recs = orc.qjl_quantize_batch(tb, dim, 42, 5, orc.lcg_normal_vecs(50, dim, 50))
    dev = [_dev(r.view(np.int16) if r.dtype == np.uint16 else r) for r in recs]
    ctx = tq.qjl_query_context(_dev(orc.lcg_normal_vecs(7, dim, 19)), 42, 5)
    ref = tq.qjl_scores(ctx, *dev, tb - 1, 42).double()
    got = tq.qjl_scores(ctx * 2.0**-122, *dev, tb - 1, 42).double() * 2.0**122
    assert ((got - ref).abs() <= 1e-6 * ref.square().mean(1, keepdim=True).sqrt()).all()


@pytest.mark.parametrize("dim,pb,nv,nq", [(128, 2, 1, 1), (128, 3, 255, 17), (64, 3, 257, 16), (32, 2, 770, 5),
                                          (32, 3, 4100, 3), (64, 2, 4352, 33)])
def test_weighted_values_at_chunk_edges(tq, dim, pb, nv, nq):
    packed, scales = orc.quantize_vec_batch(pb, dim, 42, orc.lcg_normal_vecs(3 + nv, dim, nv))
    w = np.random.default_rng(nv).random((nq, nv)).astype(np.float32)
    got = tq.qjl_weighted_values(_dev(packed), _dev(scales.view(np.int16)), _dev(w), pb, dim, 42).cpu().numpy()
    vals = orc.dequantize_vec_batch(pb, dim, 42, packed, scales).astype(np.float64)
    bound = 1e-5 * (w.astype(np.float64) @ np.abs(vals)).max()
    assert np.abs(got - w.astype(np.float64) @ vals).max() <= bound


@pytest.mark.parametrize("rows,cols", [(3, 1), (2, 1023), (2, 1025), (1, 16384), (2, 16385), (1, 20000)])
def test_softmax_column_edges(tq, rows, cols):
    s = np.random.default_rng(cols).standard_normal((rows, cols)).astype(np.float32) * 5
    s[0, cols // 2] = -np.inf if cols > 1 else 0.0
    p = tq.softmax_rows(_dev(s), 0.5).cpu().numpy()
    z = 0.5 * s.astype(np.float64)
    ref = np.exp(z - z.max(1, keepdims=True))
    ref /= ref.sum(1, keepdims=True)
    assert (np.abs(p - ref).max(1) <= 1e-6 * ref.max(1)).all()
