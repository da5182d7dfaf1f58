"""Decode launches on both sides of the lines between 4- and 8-wave
workgroups and between 64 and 128 tokens per wave, for 4 and 8 query heads per
KV head and head_dim 256, whose 8-wave workgroups take more than 64 KiB of
LDS: against dense attention over the oracle's records, within 1e-3 as every
decode test."""
import math

import numpy as np
import pytest

from oracle import oracle as orc
from test_gpu_decode_shapes import TOL, _decode, _records, tq  # noqa: F401
from tq_testdata import bf16_round

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d,bits,nr,t", [
    (256, 3, 4, 255), (256, 4, 8, 256), (256, 4, 4, 257), (256, 3, 8, 513), (256, 3, 2, 511), (256, 4, 1, 1025),
    (128, 4, 4, 512), (128, 3, 4, 513), (128, 3, 8, 1024), (128, 4, 8, 1025), (64, 3, 8, 65), (64, 4, 8, 2049),
    (256, 3, 4, 512), (256, 4, 4, 2000), (256, 3, 8, 16384), (256, 3, 4, 16385), (256, 4, 4, 16382),
])
def test_workgroup_size_edges(tq, d, bits, nr, t):  # noqa: F811
    hkv = 2
    rng = np.random.default_rng(d + bits + 10 * nr + t)
    recs, _, kd, vd = _records(rng, hkv, t, t + 3, d, bits)
    q = bf16_round(rng.standard_normal((hkv * nr, d)).astype(np.float32) / np.float32(math.sqrt(d)))
    ref = orc.attention_dense(q, kd, vd, 1 / math.sqrt(d))
    # the capacity decides the launch: exactly t, then room for more
    for cap in (t, t + 3):
        r = [x[:, :cap].contiguous() for x in recs]
        assert np.abs(_decode(tq, q, r, hkv, t, cap, d, bits) - ref).max() <= TOL
