"""The TQ cache's logit bias on the matrix cores against a float64 sum, at the
edges of its tiles: 16- and 64-row blocks, 64- and 512-token blocks, rows of
the output that start on no 4-element boundary, each source (rq given, or
R q of f32, bf16 and f16 queries formed in the launch) and output type.

Tolerance: rq enters as two f16 parts that keep 22 of its significant bits
relative to each element (2^-22), the f32 sum of D terms is off by at most
D 2^-24 of the terms' magnitudes; both are bounded by sum |rq| 2^-16 (D <= 256).
A 16-bit output adds half an ulp of its own (2^-8 for bf16, 2^-11 for f16).
"""
import numpy as np
import pytest

from oracle import oracle as orc

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

ULP = {"f32": 2.0 ** -23, "bf16": 2.0 ** -8, "f16": 2.0 ** -11}


@pytest.fixture(scope="module")
def tq():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import turboquant_amd
    return turboquant_amd


def _bias64(rq, signs, norms, d):
    """(bias, sum |rq| |c|) in f64 for rq [Hk, rows, d], signs [Hk, T, d/8], norms [Hk, T] f16."""
    b = np.unpackbits(signs, axis=-1, bitorder="little").astype(np.float64) * 2 - 1
    c = np.abs(norms.astype(np.float64)) * (np.sqrt(np.pi / 2) / np.sqrt(d))
    ref = (rq.astype(np.float64) @ b.transpose(0, 2, 1)) * c[:, None, :]
    return ref, np.abs(rq.astype(np.float64)).sum(-1)[:, :, None] * c[:, None, :]


@pytest.mark.parametrize("d,heads,q_len,kv_len,dtype", [
    (128, 2, 1, 1, "f32"), (128, 4, 3, 63, "bf16"), (64, 2, 16, 64, "f16"), (64, 6, 11, 65, "f32"),
    (128, 2, 65, 511, "bf16"), (256, 2, 17, 513, "f32"), (128, 8, 16, 1030, "f16"), (256, 4, 40, 260, "bf16"),
    (64, 4, 2, 257, "f32"), (256, 6, 1, 1025, "bf16"), (64, 64, 1, 16385, "f16"), (256, 2, 4, 16384, "f32"), (64, 2, 300, 6700, "bf16"),
    (128, 4, 3, 129, "f32"), (256, 2, 70, 127, "f16"), (128, 2, 200, 4000, "f32"), (64, 32, 4, 1000, "f32"),
    (64, 4, 2, 131073, "bf16"), (128, 2, 3, 131075, "f32"), (256, 8, 1, 131072, "f16"), (128, 8, 1, 131073, "f32"),
])
def test_bias_of_given_projections(tq, d, heads, q_len, kv_len, dtype):
    hk = 2
    rng = np.random.default_rng(kv_len)
    rq = rng.standard_normal((heads, q_len, d)).astype(np.float32)
    rq[0] *= 1e-20
    rq[-1, -1] *= 1e20
    stride = kv_len + 3
    signs = rng.integers(0, 256, (hk, stride, d // 8), dtype=np.uint8)
    norms = np.abs(rng.standard_normal((hk, stride))).astype(np.float16)
    norms[:, 0] = 0
    out = tq.qjl_logit_bias(torch.from_numpy(rq).cuda(), torch.from_numpy(signs).cuda(),
                            torch.from_numpy(norms.view(np.int16)).cuda(), hk, kv_len, stride,
                            {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}[dtype])
    ref, mag = _bias64(rq.reshape(hk, -1, d), signs[:, :kv_len], norms[:, :kv_len], d)
    got = out.float().cpu().numpy().astype(np.float64).reshape(ref.shape)
    fits = np.abs(ref) < (6e4 if dtype == "f16" else 3e38)
    err = np.abs(got - ref)[fits]
    tol = (mag * 2.0 ** -16 + np.abs(ref) * ULP[dtype] + (2.0 ** -25 if dtype == "f16" else 1e-37))[fits]
    assert (err <= tol).all(), float((err / tol).max())


def test_infinite_and_nan_projections(tq):
    d, kv = 128, 70
    rng = np.random.default_rng(9)
    rq = rng.standard_normal((1, 4, d)).astype(np.float32)
    rq[0, 1, 5] = np.inf
    rq[0, 2, 7] = np.nan
    signs = rng.integers(0, 256, (1, kv, d // 8), dtype=np.uint8)
    norms = np.ones((1, kv), np.float16)
    got = tq.qjl_logit_bias(torch.from_numpy(rq).cuda(), torch.from_numpy(signs).cuda(),
                            torch.from_numpy(norms.view(np.int16)).cuda(), 1, kv, kv).cpu().numpy()[0]
    bit = np.unpackbits(signs[0], axis=-1, bitorder="little")[:, 5]
    assert np.isfinite(got[[0, 3]]).all() and np.isnan(got[2]).all()
    assert (got[1] == np.where(bit, np.inf, -np.inf)).all()


@pytest.mark.parametrize("d,hq,t,q_len,dtype,skew", [
    (64, 4, 33, 5, "f16", 0), (128, 2, 70, 1, "f32", 0), (128, 4, 64, 33, "bf16", 0), (256, 4, 20, 18, "f32", 0),
    (128, 4, 40, 3, "bf16", 1), (256, 2, 16385, 2, "f32", 0),
])
def test_bias_of_queries_in_the_cache(tq, d, hq, t, q_len, dtype, skew):
    """skew: the queries start one element past a 16-byte boundary, which takes the launch that reads rq."""
    hk = 2
    dt = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}[dtype]
    g = torch.Generator(device="cuda").manual_seed(t)
    k, v = (torch.randn((1, hk, t, d), generator=g, device="cuda").to(dt) for _ in range(2))
    buf = torch.randn((hq * q_len * d + 8,), generator=g, device="cuda").to(dt)
    q = buf[skew:skew + hq * q_len * d].view(1, hq, q_len, d)
    cache = tq.TqCache(tq.CacheConfig(bits=3, head_dim=d, num_kv_heads=hk, num_layers=1, outlier_blocks=0))
    bias = cache.prefill(0, k, v, q).logit_bias
    signs, norms = (x.cpu().numpy() for x in cache.read_qjl(0))
    rows = np.stack([orc.rademacher_row(d, 12345, j) for j in range(d)]).astype(np.float64)
    rq = q[0].double().cpu().numpy() @ np.sign(rows).T / np.sqrt(d)
    ref, mag = _bias64(rq.reshape(hk, -1, d), signs, norms.view(np.float16), d)
    # the projection's own f32 sum: D 2^-24 of sum |q|, through D signs
    mag = mag + (np.abs(q[0].double().cpu().numpy()).sum(-1).reshape(hk, -1, 1) * np.sqrt(d) *
                 np.abs(norms.view(np.float16).astype(np.float64))[:, None, :])
    got = bias.float().cpu().numpy().astype(np.float64).reshape(ref.shape)
    err = np.abs(got - ref)
    tol = mag * 2.0 ** -16 + np.abs(ref) * ULP[dtype] + (2.0 ** -25 if dtype == "f16" else 0)
    assert (err <= tol).all(), float((err / tol).max())


@pytest.mark.parametrize("d", [64, 128, 256])
def test_bias_of_tiny_queries(tq, d):
    """Projections times 2^-122 and f32 queries times 2^-118 give the bias times the same: their elements are rounded
    to 2^-149 (2^-27 of them) and each output once more (2^-24), 1e-6 of the row's root mean square.  Rows on a
    clamped scale or cut into parts below f32's normal range are off by 1e-5 and more."""
    hk, hq, t, q_len = 2, 4, 70, 21
    g = torch.Generator(device="cuda").manual_seed(d)
    k, v = (torch.randn((1, hk, t, d), generator=g, device="cuda") for _ in range(2))
    q = torch.randn((1, hq, q_len, d), generator=g, device="cuda")
    caches = [tq.TqCache(tq.CacheConfig(bits=3, head_dim=d, num_kv_heads=hk, num_layers=1, outlier_blocks=0)) for _ in range(2)]
    pairs = [(caches[0].prefill(0, k, v, q).logit_bias[0], caches[1].prefill(0, k, v, q * 2.0**-118).logit_bias[0], 118)]
    rec = (*caches[0].read_qjl(0), hk, t, t)
    pairs.append((tq.qjl_logit_bias(q[0], *rec), tq.qjl_logit_bias(q[0] * 2.0**-122, *rec), 122))
    for ref, got, e in pairs:
        ref, got = ref.double(), got.double() * 2.0**e
        assert ((got - ref).abs() <= 1e-6 * ref.square().mean(-1, keepdim=True).sqrt()).all(), e
