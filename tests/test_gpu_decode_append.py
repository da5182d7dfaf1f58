"""A one-token decode, whose launch stores the token before it
attends: records equal to polar_quantize's and outputs equal, bit for bit, to
a decode over records that an append of its own has stored, at the edges of
the chunks (one workgroup per KV head, several, a token that opens a chunk),
for every dtype, both bit widths and codebooks, 1 to 16 query heads per KV
head and growth in between."""
import math

import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


@pytest.fixture(scope="module")
def tq():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import turboquant_amd
    return turboquant_amd


@pytest.mark.parametrize("d,bits,pq,hkv,nr,dtype,before", [
    (128, 3, False, 8, 2, "bf16", (0, 76, 511, 512, 1023, 1024, 5000)), (128, 4, False, 2, 4, "f16", (0, 512, 1024, 2047)),
    (128, 3, True, 2, 8, "f32", (1, 513)), (64, 4, True, 3, 1, "bf16", (63, 512)), (256, 4, False, 2, 8, "f32", (255, 256)),
    (256, 3, False, 1, 3, "bf16", (130, 1024)), (32, 3, False, 2, 2, "f16", (9, 700)), (128, 3, False, 1, 16, "bf16", (40,)),
])
def test_token_stored_in_the_decode_launch(tq, d, bits, pq, hkv, nr, dtype, before):
    dt = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}[dtype]
    ob = 0 if pq else tq.cache.OUTLIER_ALL
    cfg = tq.CacheConfig(bits=bits, head_dim=d, num_kv_heads=hkv, num_layers=1, outlier_blocks=ob)
    att = tq.AttendConfig(1 / math.sqrt(d), nr)
    g = torch.Generator(device="cuda").manual_seed(d + bits + nr)
    for t in before:
        k, v = (torch.randn((1, hkv, t + 2, d), generator=g, device="cuda").to(dt) for _ in range(2))
        q = torch.randn((1, hkv * nr, 2, d), generator=g, device="cuda").to(dt)
        one, two = tq.PqoCache(cfg), tq.PqoCache(cfg)
        if t:
            for c in (one, two):
                c.prefill(0, k[:, :, :t].contiguous(), v[:, :, :t].contiguous())
        for i in range(2):
            s = slice(t + i, t + i + 1)
            ki, vi, qi = k[:, :, s].contiguous(), v[:, :, s].contiguous(), q[:, :, i:i + 1].contiguous()
            got = one.decode(0, ki, vi, qi, att)
            two.decode_dequantized(0, ki, vi)  # stores with a launch of its own
            none = torch.empty((1, hkv, 0, d), dtype=dt, device="cuda")
            ref = two.decode(0, none, none, qi, att)
            assert torch.equal(got, ref), (t, i)
            assert one.seq_len(0) == two.seq_len(0) == t + i + 1
        for a, b in zip(one.read_layer(0), two.read_layer(0)):
            assert torch.equal(a, b)
        p, sc = tq.polar_quantize(k.reshape(-1, d), bits, ob)
        ki, ks, _, _ = one.read_layer(0)
        assert torch.equal(ki.view(p.shape), p) and torch.equal(ks.view(sc.shape), sc)


@pytest.mark.parametrize("d,bits,hkv,nr,dtype,before", [
    (128, 3, 8, 2, "bf16", (0, 76, 511, 1024)), (128, 4, 2, 4, "f16", (512, 2047)), (64, 4, 2, 4, "f32", (63, 512, 1030)),
    (64, 3, 3, 1, "bf16", (9,)), (256, 3, 1, 2, "f32", (255, 256)), (256, 4, 2, 8, "f16", (130,)), (128, 3, 1, 16, "bf16", (40,)),
])
def test_tq_token_stored_and_sketched_in_the_decode_launch(tq, d, bits, hkv, nr, dtype, before):
    """Records, signs and norms as a prefill of the same tokens stores them; the output equals that of a decode over
    them, which projects the query in the launch too."""
    dt = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}[dtype]
    cfg = tq.CacheConfig(bits=bits, head_dim=d, num_kv_heads=hkv, num_layers=1, outlier_blocks=0)
    att = tq.AttendConfig(1 / math.sqrt(d), nr)
    g = torch.Generator(device="cuda").manual_seed(d + bits + nr)
    for t in before:
        k, v = (torch.randn((1, hkv, t + 1, d), generator=g, device="cuda").to(dt) for _ in range(2))
        q = torch.randn((1, hkv * nr, 1, d), generator=g, device="cuda").to(dt)
        one, two = tq.TqCache(cfg), tq.TqCache(cfg)
        if t:
            one.prefill(0, k[:, :, :t].contiguous(), v[:, :, :t].contiguous(), q)
        got = one.decode(0, k[:, :, t:].contiguous(), v[:, :, t:].contiguous(), q, att)
        two.prefill(0, k, v, q)
        none = torch.empty((1, hkv, 0, d), dtype=dt, device="cuda")
        ref = two.decode(0, none, none, q, att)
        for a, b in zip((*one.read_layer(0), *one.read_qjl(0)), (*two.read_layer(0), *two.read_qjl(0))):
            assert torch.equal(a, b), t
        if nr <= 8:
            assert torch.equal(got, ref), t
        else:  # several head groups: the append's own launch projects q, in another order of its f32 sums (1e-5): an ulp
            a, b = got.float(), ref.float()
            assert ((a - b).abs() <= 2.0**-7 * b.abs() + 1e-5 * b.abs().max()).all()


@pytest.mark.parametrize("kind,norm,d,bits,hkv,nr,before", [
    ("tq", 0, 128, 3, 2, 16, (40, 700)), ("tq", 1, 128, 3, 2, 2, (40, 1500)), ("tq", 1, 64, 4, 3, 1, (9,)),
    ("tq", 1, 256, 3, 1, 4, (300,)), ("tq", 0, 64, 3, 64, 1, (7000,)), ("tq", 0, 128, 4, 64, 2, (7000,)),
    ("pqo", 0, 64, 3, 64, 1, (2000, 7000)), ("pqo", 0, 64, 4, 64, 2, (7000,)), ("pq", 0, 64, 4, 64, 1, (7000,)),
    ("pqo", 1, 64, 3, 64, 1, (7000,)), ("pq", 0, 128, 3, 2, 16, (700,)),
])
def test_token_stored_by_a_launch_of_its_own(tq, kind, norm, d, bits, hkv, nr, before):
    """More than 8 query heads per KV head, L2Norm, and contexts that take range launches (64 KV heads x 7,000 tokens):
    the records as a prefill stores them, the output bit for bit that of a decode over them given rq = R q."""
    ob = tq.cache.OUTLIER_ALL if kind == "pqo" else 0
    cfg = tq.CacheConfig(bits, d, hkv, 1, tq.cache.QuantNormMode(norm), ob)
    make = tq.TqCache if kind == "tq" else tq.PqoCache
    lib, check = tq._lib.lib, tq._lib.check
    g = torch.Generator(device="cuda").manual_seed(d + nr)
    for t in before:
        k, v = (torch.randn((1, hkv, t + 1, d), generator=g, device="cuda") for _ in range(2))
        q = torch.randn((1, hkv * nr, 1, d), generator=g, device="cuda")
        one, two = make(cfg), make(cfg)
        one.prefill(0, k[:, :, :t].contiguous(), v[:, :, :t].contiguous(), q)
        got = one.decode(0, k[:, :, t:].contiguous(), v[:, :, t:].contiguous(), q, tq.AttendConfig(d**-0.5, nr))
        two.prefill(0, k, v, q)
        read = lambda c: (*c.read_layer(0), *(c.read_qjl(0) if kind == "tq" else ()))
        for a, b in zip(read(one), read(two)):
            assert torch.equal(a, b), t
        # decode over the records of `one`, whose capacity sets the split
        cap, rq = one.capacity(0), None
        if kind == "tq":
            rq = tq.qjl_project(q.view(-1, d), tq.qjl_sign_matrix(d, tq.cache.DEFAULT_QJL_SEED))
        ki, ks, vi, vs, sg, nm = one.buffers(0)
        ws = tq.AttentionWorkspace(1, hkv * nr, hkv, d, cap)
        lens = torch.tensor([t + 1], dtype=torch.int32, device="cuda")
        out = torch.empty_like(q)
        check(lib.tq_cache_decode_attention(
            q.data_ptr(), 0, ki, ks, vi, vs, rq.data_ptr() if kind == "tq" else None, sg, nm, lens.data_ptr(), 1, hkv * nr,
            hkv, d, bits, ob, norm, cap, cap, hkv * cap, d**-0.5, out.data_ptr(), 0, ws.buf.data_ptr(), ws.nbytes,
            torch.cuda.current_stream().cuda_stream))
        assert torch.equal(got, out), t


def test_a_refused_shape_still_stores_its_token(tq):
    cfg = tq.CacheConfig(bits=3, head_dim=96, num_kv_heads=2, num_layers=1)
    c = tq.PqoCache(cfg)
    k = torch.randn((1, 2, 1, 96), device="cuda")
    with pytest.raises(tq.TurboQuantError, match="head_dim 32, 64, 128 or 256"):
        c.decode(0, k, k, k, tq.AttendConfig(0.1, 1))
    assert c.seq_len(0) == 1
    p, _ = tq.polar_quantize(k.reshape(-1, 96), 3)
    assert torch.equal(c.read_layer(0)[0].view(p.shape), p)
