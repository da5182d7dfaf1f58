"""A layer that grows while records of every size are in it (copied in units
of 2 to 16 bytes): what is stored equals one quantize of the whole, and the
capacity past it is zero."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


@pytest.fixture(scope="module")
def tq():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import turboquant_amd
    return turboquant_amd


@pytest.mark.parametrize("d,bits,heads,qjl,pieces", [
    (32, 3, 3, False, (1, 200, 3)), (96, 3, 2, False, (5, 131)), (64, 3, 1, True, (7, 150, 1)),
    (128, 3, 8, True, (1, 128, 40)), (128, 4, 5, False, (300, 77)), (256, 4, 2, True, (3, 129)),
])
def test_growth_keeps_records_and_zeroes_the_rest(tq, d, bits, heads, qjl, pieces):
    ob = 0 if qjl else tq.cache.OUTLIER_ALL
    cfg = tq.CacheConfig(bits=bits, head_dim=d, num_kv_heads=heads, num_layers=2, outlier_blocks=ob)
    cache = (tq.TqCache if qjl else tq.PqoCache)(cfg)
    g = torch.Generator(device="cuda").manual_seed(d + bits)
    t = sum(pieces)
    k, v = (torch.randn((1, heads, t, d), generator=g, device="cuda") for _ in range(2))
    q = torch.randn((1, heads, 1, d), generator=g, device="cuda")
    at = 0
    for n in pieces:
        cache.prefill(1, k[:, :, at:at + n].contiguous(), v[:, :, at:at + n].contiguous(), q)
        at += n
    ki, ks, vi, vs = cache.read_layer(1)
    for x, idx, sc in ((k, ki, ks), (v, vi, vs)):
        p, s = tq.polar_quantize(x.reshape(-1, d), bits, ob)
        assert torch.equal(idx.view(p.shape), p) and torch.equal(sc.view(s.shape), s)
    if qjl:
        whole = tq.TqCache(cfg)
        whole.prefill(1, k, v, q)
        assert all(torch.equal(a, b) for a, b in zip(cache.read_qjl(1), whole.read_qjl(1)))
    # the capacity past the stored rows, through the raw buffers
    cap = cache.capacity(1)
    assert cap > t
    hip = C.CDLL("libamdhip64.so")
    for ptr, rec in zip(cache.buffers(1), (d * bits // 8, d // 16, d * bits // 8, d // 16, d // 8, 2)):
        if ptr is None:
            continue
        host = np.empty((heads, cap, rec), np.uint8)
        torch.cuda.synchronize()
        assert hip.hipMemcpy(host.ctypes.data_as(C.c_void_p), C.c_void_p(ptr), C.c_size_t(host.nbytes), 2) == 0
        assert not host[:, t:].any() and host[:, :t].any()
