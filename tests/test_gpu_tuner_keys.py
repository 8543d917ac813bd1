"""The tuner keeps apart what it times differently: sets of one shape whose sticks are
runs or not (z addressing to choose or none), and small sets whose values the backward
matrix kernel takes itself or not (a z kernel less). In a fresh process, since the choices
are per process: the set with less to choose from comes first, and the other one is still
timed on its first call. Single transforms and batches of two."""
import os
import subprocess
import sys

import pytest

pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

CHILD = r'''
import sys
sys.path.insert(0, sys.argv[1])
import numpy as np
import torch
import spfft_amd as sp
from tests.test_gpu_matrix import ellipsoid
from tests.test_gpu_parity import build

def shells(t):
    return np.ascontiguousarray(t[np.argsort((t.astype(int) ** 2).sum(1), kind="stable")])

def longer(t, n):
    # every stick near the axis over all z: the same sticks, more values
    inner = {(x, y) for x, y, z in t.tolist() if x * x + y * y <= 9}
    rest = [k for k in t.tolist() if (k[0], k[1]) not in inner]
    more = [[x, y, z] for x, y in inner for z in range(-(n // 2) + 1, n // 2)]
    return np.array(sorted(rest + more), np.int32)

small = ellipsoid((32, 32, 32), 0.27)
assert len(small) <= 3000 < len(longer(small, 32))
pairs = [((48, 48, 48), shells(ellipsoid((48, 48, 48), 0.3)), ellipsoid((48, 48, 48), 0.3)),
         ((32, 32, 32), longer(small, 32), small)]
for dims, first, second in pairs:
    for t in (first, second):
        for count in (1, 2):
            trs = [build(dims, t, False, "double") for _ in range(count)]
            ins = [torch.zeros(2 * len(t), dtype=torch.float64, device="cuda") for _ in trs]
            outs = [torch.empty(2 * int(np.prod(dims)), dtype=torch.float64, device="cuda")
                    for _ in trs]
            if count == 1:
                trs[0].backward(ins[0], outs[0])
            else:
                sp.multi_transform_backward(trs, ins, outs)
            torch.cuda.synchronize()
print("child done", flush=True)
'''


def test_sets_of_one_shape_are_timed_apart(tmp_path):
    env = dict(os.environ, SPFFT_AMD_TUNE_CACHE="off", SPFFT_AMD_TUNE_LOG="1")
    env.pop("SPFFT_AMD_PLANE", None)
    script = tmp_path / "child.py"
    script.write_text(CHILD)
    print("tuner keys", flush=True)
    r = subprocess.run([sys.executable, "-u", str(script), ROOT], env=env, capture_output=True,
                       text=True, timeout=100, cwd=ROOT)
    assert r.returncode == 0, r.stdout + r.stderr
    lines = [ln for ln in r.stderr.splitlines() if ln.startswith("spfft_amd tune:")]
    assert len(lines) == 8, r.stderr
