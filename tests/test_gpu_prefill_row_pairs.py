"""Staged prefill tiles whose waves work in pairs, each pair on 32 rows and
each wave of it on half of every tile: halves that no row sees (sequences and
causal rows that end in a tile's first half), ragged last rows of a pair, and
rows whose two halves hold very different maxima, and the shorter walks that
waves take one group each, against the oracle in double.  Tolerance 1e-3 max-abs, as for every prefill (fp32 accumulation, f16
two-part operands)."""
import math

import numpy as np
import pytest

from oracle import oracle as orc
from tq_testdata import bf16_bits, bf16_round, kv_outlier

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

D = 128


def _dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


@pytest.mark.parametrize("bits,outlier,hq,hkv,ql,t,causal,peak,splits", [
    # walks of at least 24 tiles: pairs
    (3, orc.OUTLIER_ALL, 2, 1, 1, 1536 + 20, True, None, 1),    # nothing in the last tile's second half
    (4, orc.OUTLIER_ALL, 4, 1, 9, 1472 + 32, False, None, 1),   # 24 tiles, the last one's second half is empty
    (3, 0, 2, 2, 1475, 1475, True, None, 1),                    # causal rows that see one half only; ragged rows
    (4, 0, 1, 1, 130, 3073, True, None, 2),                     # two splits of 25 tiles, one row of a second workgroup
    (3, orc.OUTLIER_ALL, 1, 1, 65, 1568, False, 5, 1),          # the maximum in a first half
    (3, orc.OUTLIER_ALL, 1, 1, 65, 1568, False, 64 + 40, 1),    # and in a second half
    # shorter walks: one group per wave
    (4, 0, 4, 1, 9, 1472, False, None, 1),                      # 23 tiles
    (3, orc.OUTLIER_ALL, 2, 1, 1, 768 + 20, True, None, 1),
    (4, orc.OUTLIER_ALL, 4, 1, 9, 704 + 32, False, None, 1),
    (4, 0, 4, 1, 9, 704, False, None, 1),
    (3, 0, 2, 2, 707, 707, True, None, 1),
    (4, 0, 1, 1, 130, 1601, True, None, 2),
    (3, orc.OUTLIER_ALL, 1, 1, 65, 800, False, 5, 1),
    (3, orc.OUTLIER_ALL, 1, 1, 65, 800, False, 64 + 40, 1),
])
@pytest.mark.parametrize("qdt", ["bf16", "f32"])
def test_staged_row_pairs(monkeypatch, bits, outlier, hq, hkv, ql, t, causal, peak, splits, qdt):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import turboquant_amd as tq
    rng = np.random.default_rng(4100 + 7 * t + ql)
    k, v = kv_outlier(rng, hkv, t), kv_outlier(rng, hkv, t)
    q = rng.standard_normal((hq, ql, D)).astype(np.float32) / np.float32(math.sqrt(D))
    scale = 1 / math.sqrt(D)
    if peak is not None:
        k[:, peak] = 30.0 * q[0, 0] / np.linalg.norm(q[0, 0])
        q[:] = q[0, 0] * 20.0
    q = bf16_round(q)
    recs, deq = [], []
    for x in (k, v):
        p, s = orc.polar_quantize(bits, outlier, x.reshape(-1, D), D)
        deq.append(orc.polar_dequantize(bits, outlier, p, s, D).reshape(hkv, t, D))
        recs += [_dev(p.reshape(hkv, t, -1)), _dev(s.reshape(hkv, t, 4).view(np.int16))]
    qd = _dev(bf16_bits(q)).view(torch.bfloat16) if qdt == "bf16" else _dev(q)
    monkeypatch.setenv("TQ_PREFILL_STAGING", "1")
    monkeypatch.setenv("TQ_PREFILL_SPLITS", str(splits))
    out = tq.cache_prefill_attention(qd, recs[0], recs[1], recs[2], recs[3], hkv, bits, t, t, scale, outlier,
                                     causal=causal)
    torch.cuda.synchronize()
    ref = orc.attention_prefill(q, deq[0], deq[1], scale, causal)
    err = np.abs(out.float().cpu().numpy() - ref).max()
    assert err <= 1e-3, err
