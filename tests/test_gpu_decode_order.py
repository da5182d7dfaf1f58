"""The split of a long context over workgroups depends on its own launch
alone: outputs are the same bits whichever decode the process ran before.  The
L2Norm and MaxNorm kernels of 4-bit PQO at head_dim 256 with 8 query heads per
KV head differ in how many workgroups a compute unit holds."""
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CHILD = """
import hashlib, sys, torch
import turboquant_amd as tq
for norm in map(int, sys.argv[1:]):
    g = torch.Generator(device="cuda").manual_seed(7)
    k, v = (torch.randn((1, 64, 3401, 256), generator=g, device="cuda") for _ in range(2))
    q = torch.randn((1, 512, 1, 256), generator=g, device="cuda")
    c = tq.PqoCache(tq.CacheConfig(4, 256, 64, 1, tq.cache.QuantNormMode(norm)))
    c.prefill(0, k[:, :, 1:].contiguous(), v[:, :, 1:].contiguous())
    out = c.decode(0, k[:, :, :1].contiguous(), v[:, :, :1].contiguous(), q, tq.AttendConfig(0.0625, 8))
    print(norm, hashlib.sha256(out.cpu().numpy().tobytes()).hexdigest())
"""


def test_split_does_not_depend_on_earlier_launches():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    seen = [sorted(subprocess.run([sys.executable, "-c", CHILD, *order], capture_output=True, text=True, check=True,
                                  timeout=100, cwd=ROOT).stdout.splitlines()) for order in (("0", "1"), ("1", "0"))]
    assert len(seen[0]) == 2 and seen[0] == seen[1]
