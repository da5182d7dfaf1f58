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


@pytest.mark.parametrize("dim,tb,nk,nq", [(32, 3, 5, 1), (32, 3, 32769, 2), (32, 3, 33000, 17), (64, 4, 49153, 1),
                                          (128, 3, 24577, 1), (128, 4, 33007, 3)])
def test_scores_of_many_keys(tq, dim, tb, nk, nq):
    """Lists at which a wave walks several tiles of 16 keys, and few queries by tables: against the oracle on some
    hundred of the keys, which are all that the list repeats."""
    part = orc.lcg_normal_vecs(dim + nk, dim, 211)
    recs = orc.qjl_quantize_batch(tb, dim, 42, 5, part)
    qs = orc.lcg_normal_vecs(nq, dim, nq)
    ref = orc.qjl_scores(tb - 1, dim, 42, 5, qs, *recs)
    at = np.arange(nk) % len(part)
    dev = [_dev((r.view(np.int16) if r.dtype == np.uint16 else r)[at]) for r in recs]
    got = tq.qjl_scores(tq.qjl_query_context(_dev(qs), 42, 5), *dev, tb - 1, 42).cpu().numpy()
    natural = np.linalg.norm(qs, axis=1)[:, None] * np.linalg.norm(part, axis=1)[None, :]
    assert (np.abs(got - ref[:, at]) / natural[:, at]).max() <= 1e-5


@pytest.mark.parametrize("nk,nq,gib", [(2**29 + 1, 2, 16), (2**32 + 1, 1, 100)])
def test_scores_of_more_keys_than_one_launch_holds(tq, nk, nq, gib):
    """A launch holds fewer than 2^32 lanes: eight or one a key.  The last key's score is that of the key alone."""
    dim = 32
    if torch.cuda.mem_get_info()[0] < gib * 2**30:
        pytest.skip(f"needs {gib} GiB")
    recs = [torch.zeros((nk, 8), dtype=torch.uint8, device="cuda"), torch.zeros((nk,), dtype=torch.int16, device="cuda"),
            torch.zeros((nk, 4), dtype=torch.uint8, device="cuda"), torch.zeros((nk,), dtype=torch.int16, device="cuda")]
    last = [_dev(r.view(np.int16) if r.dtype == np.uint16 else r)
            for r in orc.qjl_quantize_batch(3, dim, 42, 5, orc.lcg_normal_vecs(1, dim, 1))]
    for r, x in zip(recs, last):
        r[-1:] = x
    ctx = tq.qjl_query_context(_dev(orc.lcg_normal_vecs(2, dim, nq)), 42, 5)
    got = tq.qjl_scores(ctx, *recs, 2, 42)
    ref = tq.qjl_scores(ctx, *last, 2, 42)[0].cpu()  # by tables or products as the list's length has it
    del recs, r
    assert torch.allclose(got[0, -1:].cpu(), ref, rtol=1e-5) and float(ref) != 0.0 and float(got[0, 5]) == 0.0
    del got
    torch.cuda.empty_cache()


def test_sketch_of_more_vectors_than_one_launch_holds(tq):
    """2^28 + 1 vectors of 128: 512 lanes for 32 of them, and a launch holds fewer than 2^32.  The first and the last
    one's records are those of the vector alone."""
    n, dim = 2**28 + 1, 128
    if torch.cuda.mem_get_info()[0] < 200 * 2**30:
        pytest.skip("needs 200 GiB")
    one = _dev(orc.lcg_normal_vecs(1, dim, 1))
    x = torch.zeros((n, dim), device="cuda")
    x[0], x[-1] = one[0], one[0]
    ref = tq.qjl_quantize_batch(one, 3, 42, 5)
    got = tq.qjl_quantize_batch(x, 3, 42, 5)
    del x
    try:
        for r, g in zip(ref, got):
            assert torch.equal(g[0], r[0]) and torch.equal(g[-1], r[0])
    finally:
        del got, g
        torch.cuda.empty_cache()


def test_scores_of_infinite_and_nan_queries(tq):
    """Rows with an infinity or a NaN are not finite, as the oracle's; the other rows of their tile keep their values,
    huge and tiny ones too; a key whose scale overflows f16 is not finite for any query."""
    dim, tb, nk = 64, 4, 40
    keys, qs = orc.lcg_normal_vecs(3, dim, nk), orc.lcg_normal_vecs(4, dim, 7)
    keys[11] *= 1e6
    qs[1, 5], qs[2, 9] = np.inf, np.nan
    qs[3] *= 1e30
    qs[4] *= 1e-30
    recs = orc.qjl_quantize_batch(tb, dim, 42, 5, keys)
    with np.errstate(all="ignore"):
        ref = orc.qjl_scores(tb - 1, dim, 42, 5, qs, *recs)
    dev = [_dev(r.view(np.int16) if r.dtype == np.uint16 else r) for r in recs]
    got = tq.qjl_scores(tq.qjl_query_context(_dev(qs), 42, 5), *dev, tb - 1, 42).cpu().numpy()
    assert (np.isfinite(got) == np.isfinite(ref)).all()
    assert not np.isfinite(got[1:3]).any() and not np.isfinite(got[:, 11]).any()
    rows, cols = [0, 3, 4, 5, 6], [j for j in range(nk) if j != 11]
    natural = np.linalg.norm(qs[rows].astype(np.float64), axis=1)[:, None] * np.linalg.norm(keys[cols], axis=1)[None, :]
    assert (np.abs(got[np.ix_(rows, cols)] - ref[np.ix_(rows, cols)].astype(np.float64)) / natural).max() <= 1e-5


@pytest.mark.parametrize("dim,tb", [(32, 3), (32, 4), (64, 3), (128, 3), (128, 4)])
def test_scores_are_as_exact_as_f32_sums(tq, dim, tb):
    """Against f64, the 2-norm of the error is no larger than that of f32 sums of pairs of products and groups of four
    signed projections, which the split of the operands into f16 parts stands for."""
    nk, nq, pb = 600, 40, tb - 1
    recs = orc.qjl_quantize_batch(tb, dim, 42, 5, orc.lcg_normal_vecs(dim, dim, nk))
    packed, sc, sg, nm = [_dev(r.view(np.int16) if r.dtype == np.uint16 else r) for r in recs]
    ctx = tq.qjl_query_context(_dev(orc.lcg_normal_vecs(9, dim, nq)), 42, 5)
    got = tq.qjl_scores(ctx, packed, sc, sg, nm, pb, 42).cpu().numpy().astype(np.float64)
    unit = torch.full((nk,), 1.0, dtype=torch.float16).cuda().view(torch.int16)
    x = tq.dequantize_rotated_batch(packed, unit, pb, dim).cpu().numpy()  # the centroids
    qt, rq = ctx.cpu().numpy().reshape(nq, 2, dim).transpose(1, 0, 2)
    bits = np.unpackbits(sg.cpu().numpy(), axis=-1, bitorder="little").astype(np.float32) * 2 - 1
    scale, norm = recs[1].view(np.float16).astype(np.float32), recs[3].view(np.float16).astype(np.float32)

    def sums(dt):
        a, b = (np.asarray(z, dt) for z in (qt[:, None, :] * x.astype(dt), rq[:, None, :] * bits.astype(dt)))
        a = a[..., ::2] + a[..., 1::2]
        b = ((b[..., ::4] + b[..., 1::4]) + b[..., 2::4]) + b[..., 3::4]
        ck = norm.astype(dt) * dt(1.2533141) / np.sqrt(dt(dim))
        return scale.astype(dt) * np.cumsum(a, -1, dtype=dt)[..., -1] + ck * np.cumsum(b, -1, dtype=dt)[..., -1]
    ref = sums(np.float64)
    assert np.linalg.norm(got - ref) <= np.linalg.norm(sums(np.float32) - ref)


@pytest.mark.parametrize("dim,pb,nv,nq", [(128, 2, 1, 1), (128, 3, 255, 17), (64, 3, 257, 16), (32, 2, 770, 5),
                                          (32, 3, 4100, 3), (64, 2, 4352, 33),
                                          (32, 3, 5, 17), (64, 3, 31, 2), (128, 3, 32, 16), (64, 2, 33, 1)])
def test_weighted_values_at_chunk_edges(tq, dim, pb, nv, nq):
    packed, scales = orc.quantize_vec_batch(pb, dim, 42, orc.lcg_normal_vecs(3 + nv, dim, nv))
    w = np.random.default_rng(nv).random((nq, nv)).astype(np.float32)
    got = tq.qjl_weighted_values(_dev(packed), _dev(scales.view(np.int16)), _dev(w), pb, dim, 42).cpu().numpy()
    vals = orc.dequantize_vec_batch(pb, dim, 42, packed, scales).astype(np.float64)
    bound = 1e-5 * (w.astype(np.float64) @ np.abs(vals)).max()
    assert np.abs(got - w.astype(np.float64) @ vals).max() <= bound


def test_weighted_values_of_more_values_than_one_launch_holds(tq):
    """2^31 + 1 values of 128: 512 lanes for 256 of them.  All weight is on the first and the last one."""
    nv, dim = 2**31 + 1, 128
    if torch.cuda.mem_get_info()[0] < 120 * 2**30:
        pytest.skip("needs 120 GiB")
    packed, scales = orc.quantize_vec_batch(2, dim, 42, orc.lcg_normal_vecs(3, dim, 2))
    codes = torch.zeros((nv, dim // 4), dtype=torch.uint8, device="cuda")
    sc = torch.zeros((nv,), dtype=torch.int16, device="cuda")
    w = torch.zeros((1, nv), device="cuda")
    for i in (0, 1):
        codes[-i] = _dev(packed[i])
        sc[-i] = int(scales.view(np.int16)[i])
        w[0, -i] = 1.0 + i
    got = tq.qjl_weighted_values(codes, sc, w, 2, dim, 42).cpu().numpy()[0]
    del codes, sc, w
    torch.cuda.empty_cache()
    vals = orc.dequantize_vec_batch(2, dim, 42, packed, scales).astype(np.float64)
    assert np.abs(got - (vals[0] + 2 * vals[1])).max() <= 1e-5 * np.abs(vals).max()


def test_softmax_of_more_rows_than_one_launch_holds(tq):
    x = torch.zeros((2**22 + 1, 3), device="cuda")
    x[-1] = torch.tensor([0.0, 1.0, 2.0])
    p = tq.softmax_rows(x, 1.0)
    assert (p[:-1] == p[0]).all() and torch.allclose(p[-1].cpu(), torch.softmax(x[-1].cpu(), 0), atol=1e-6)


@pytest.mark.parametrize("rows,cols", [(3, 1), (2, 1023), (2, 1025), (1, 16384), (2, 16385), (1, 20000), (2, 1024), (3, 4096), (2, 4097)])
def test_softmax_column_edges(tq, rows, cols):
    s = np.random.default_rng(cols).standard_normal((rows, cols)).astype(np.float32) * 5
    s[0, cols // 2] = -np.inf if cols > 1 else 0.0
    p = tq.softmax_rows(_dev(s), 0.5).cpu().numpy()
    z = 0.5 * s.astype(np.float64)
    ref = np.exp(z - z.max(1, keepdims=True))
    ref /= ref.sum(1, keepdims=True)
    assert (np.abs(p - ref).max(1) <= 1e-6 * ref.max(1)).all()
