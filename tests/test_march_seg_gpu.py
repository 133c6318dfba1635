"""TN_MARCH_SEG fixes the node columns per block of the matrix apply: 64 columns a block make
51 blocks of 66 steps of a level-6 shell's 3250 columns, where the library's choice is a
block of 13 columns per CU, 15 steps: the same result in at least twice the time.  The
variable is read once per process: a child process each."""
import json
import os
import subprocess
import sys

import pytest

CHILD = """
import hashlib, json, sys, time
import numpy as np, torch
import terraneo_amd as tn
m = tn.Mesh(6, radii=np.linspace(0.55, 1.0, 65))
x = torch.linspace(-1.0, 1.0, 3 * m.N, device="cuda:0", dtype=torch.float64)
A = tn.Eps(m, torch.ones(m.N, device="cuda:0", dtype=torch.float64), 1, 1)
y = A.apply(x, torch.empty_like(x))
best = 1e9
for _ in range(5):
    torch.cuda.synchronize()
    t = time.perf_counter()
    for _ in range(20):
        A.apply(x, y)
    torch.cuda.synchronize()
    best = min(best, time.perf_counter() - t)
print(json.dumps([best, hashlib.sha256(y.cpu().numpy().tobytes()).hexdigest()]))
"""


@pytest.mark.gpu
def test_columns_per_block(cuda):
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    out = {}
    for seg in ("0", "1", "64"):  # 0: the library's choice
        env = dict(os.environ, TN_MARCH_SEG=seg, PYTHONPATH=root)
        r = subprocess.run([sys.executable, "-c", CHILD], env=env, capture_output=True, text=True, timeout=100)
        assert r.returncode == 0, r.stderr[-2000:]
        out[seg] = json.loads(r.stdout.strip().splitlines()[-1])
    assert out["0"][1] == out["1"][1] == out["64"][1]
    assert out["64"][0] >= 2.0 * out["0"][0], out
