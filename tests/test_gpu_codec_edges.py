"""The core codec and the QJL sketch at batch sizes that end inside a wave, a
workgroup or a group of 16 or 32 vectors: bit-exact against the oracle, and
nothing written past the last vector."""
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


def _x(dim, n):
    x = orc.lcg_normal_vecs(300 + dim + n, dim, n)
    x[n // 2] *= 1e-12  # norm below the codec's minimum
    return x


@pytest.mark.parametrize("n", [1, 2, 7, 16, 17, 32, 33, 64, 65, 128, 129, 256, 257, 323])
@pytest.mark.parametrize("dim,bits", [(32, 2), (64, 3), (128, 4), (256, 3)])
def test_core_codec_batch_edges(tq, dim, bits, n):
    x = _x(dim, n)
    p_ref, s_ref = orc.quantize_vec_batch(bits, dim, 42, x)
    p, s = tq.quantize_vec_batch(torch.from_numpy(x).cuda(), bits, 42)
    assert np.array_equal(p.cpu().numpy(), p_ref) and np.array_equal(s.cpu().numpy().view(np.uint16), s_ref)
    # dequantize into the front of a larger buffer: the rest stays
    buf = torch.full((n + 1, dim), 7.0, device="cuda")
    tq.lib.tq_dequantize_vec_batch(p.data_ptr(), s.data_ptr(), buf.data_ptr(), n, bits, dim, 42,
                                   torch.cuda.current_stream().cuda_stream)
    ref = orc.dequantize_vec_batch(bits, dim, 42, p_ref, s_ref)
    assert np.array_equal(buf[:n].cpu().numpy().view(np.uint32), ref.view(np.uint32)) and (buf[n] == 7.0).all()


@pytest.mark.parametrize("n", [1, 15, 17, 32, 33, 50])
@pytest.mark.parametrize("dim,tb", [(32, 4), (64, 3), (128, 3), (128, 4)])
def test_qjl_sketch_batch_edges(tq, dim, tb, n):
    x = _x(dim, n)
    x[0, 0] = -0.0
    ref = orc.qjl_quantize_batch(tb, dim, 7, 99, x)
    got = tq.qjl_quantize_batch(torch.from_numpy(x).cuda(), tb, 7, 99)
    for r, g in zip(ref, got):
        g = g.cpu().numpy()
        assert np.array_equal(g.view(np.uint16) if g.dtype == np.int16 else g, r)
