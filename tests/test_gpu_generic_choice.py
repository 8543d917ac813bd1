"""Sets with a long line, not all of fixed lengths and none with a prime factor above
13: the first call times the generic kernels against the matrix kernels and keeps the
faster (single transforms and batches), and either choice, once recorded, is the one
that runs, also for one transform in a multi-transform call. Outputs are checked against
the oracle each time.

Each part runs in a fresh process, since the choices are per process. Tolerances: those
of the generic kernels, 1e-12 (FP64) and 1e-5 (FP32)."""
import os
import re
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
from oracle import oracle as orc
from tests.test_gpu_matrix import ellipsoid
from tests.test_gpu_parity import build
from tests.test_gpu_split_lengths import kernels_run
from tests.workloads import complex_values

for dims, r2c, precision, count, multi in (((245, 24, 18), False, "double", 1, False),
                                           ((20, 18, 250), True, "float", 1, False),
                                           ((16, 308, 24), True, "double", 3, True),
                                           ((35, 288, 24), False, "float", 2, True),
                                           ((245, 24, 18), False, "double", 1, True)):
    print("case", dims, count, flush=True)
    t = ellipsoid(dims, 0.4, r2c)
    o = orc.OraclePlan(r2c, dims, t)
    n = int(np.prod(dims)) * (1 if r2c else 2)
    rd, dt, tol = ((np.float64, torch.float64, 1e-12) if precision == "double"
                   else (np.float32, torch.float32, 1e-5))
    vals = [complex_values(0x5EED1900 + k, len(t)) for k in range(count)]
    ins = [torch.from_numpy(v.view(np.float64).astype(rd)).cuda() for v in vals]
    spaces = [torch.empty(n, dtype=dt, device="cuda") for _ in vals]
    outs = [torch.empty(2 * len(t), dtype=dt, device="cuda") for _ in vals]
    trs = [build(dims, t, r2c, precision) for _ in vals]
    def run():
        if not multi:
            trs[0].backward(ins[0], spaces[0])
            trs[0].forward(spaces[0], outs[0], sp.SPFFT_FULL_SCALING)
        else:
            sp.multi_transform_backward(trs, ins, spaces)
            sp.multi_transform_forward(trs, spaces, outs, [sp.SPFFT_FULL_SCALING] * count)
        torch.cuda.synchronize()
    run()
    print("ran", *sorted(kernels_run(run)), flush=True)
    for k, v in enumerate(vals):
        want = o.backward(v)
        got = spaces[k].cpu().numpy().astype(np.float64)
        got = (got if r2c else got.view(np.complex128)).reshape(dims[::-1])
        assert orc.rel_l2(got, want) <= tol, k
        f = outs[k].cpu().numpy().astype(np.float64).view(np.complex128)
        assert orc.rel_l2(f, o.forward(got, True)) <= tol, k
'''


def run_child(tmp_path, cache):
    env = dict(os.environ, SPFFT_AMD_TUNE_CACHE=str(cache), SPFFT_AMD_TUNE_LOG="1")
    env.pop("SPFFT_AMD_PLANE", None)
    script = tmp_path / "child.py"
    script.write_text(CHILD)
    r = subprocess.run([sys.executable, "-u", str(script), ROOT], env=env, capture_output=True,
                       text=True, timeout=240, cwd=ROOT)
    assert r.returncode == 0, r.stdout + r.stderr
    return r.stderr, [ln.split()[1:] for ln in r.stdout.splitlines() if ln.startswith("ran")]


def test_either_choice_runs(tmp_path):
    cache = tmp_path / "tune.txt"
    print("generic choice: timed", flush=True)
    log, _ = run_child(tmp_path, cache)
    timed = re.findall(r"generic \(all stages\) ([0-9.]+)", log)
    assert len(timed) == 8 and all(float(ms) > 0 for ms in timed), log
    text = cache.read_text()
    for plane, stage, other in (("4", "k_z_backward", "_dft"), ("3", "_dft", "k_z_backward ")):
        print(f"generic choice: plane {plane}", flush=True)
        cache.write_text(re.sub(r"plane=\d", f"plane={plane}", text))
        log, ran = run_child(tmp_path, cache)
        assert "spfft_amd tune:" not in log, log
        assert len(ran) == 5
        for names in ran:
            names = " ".join(names) + " "
            assert stage in names and other not in names, (plane, names)
