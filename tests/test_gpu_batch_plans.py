"""More batches than the library keeps argument tables for (8), queued without waiting:
their tables are written into the memory of the least recently used ones while work that
reads those may still be queued. Small, large and small batches in turn, one of more
transforms than one table launch writes (12), then the first again. Against the FP64
oracle, and the second visit bit for bit as the first. Tolerance: 1e-12."""
import numpy as np
import pytest

import spfft_amd as sp
from oracle import oracle as orc
from tests.test_gpu_matrix import ellipsoid
from tests.test_gpu_parity import build
from tests.workloads import complex_values

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims", [(32, 32, 32), (20, 24, 18)], ids=lambda d: "x".join(map(str, d)))
def test_tables_are_replaced_in_order(dims):
    sizes = [2, 30, 3, 13, 2, 5, 12, 4, 25, 2, 3, 40]
    sets = [ellipsoid(dims, f) for f in (0.25, 0.33, 0.4)]
    plans = [orc.OraclePlan(False, dims, t) for t in sets]
    n = 2 * int(np.prod(dims))
    pool = [[build(dims, t, False, "double") for _ in range(14)] for t in sets]
    trs = [pool[k % 3][k // 3] for k in range(42)]
    for t in trs:
        t.set_execution_mode(sp.SPFFT_EXEC_ASYNCHRONOUS)
    vals = [complex_values(0x5EED1E00 + k, len(sets[k % 3])) for k in range(42)]
    ins = [torch.from_numpy(v.view(np.float64)).cuda() for v in vals]
    batches = []
    for b, size in enumerate(sizes):
        at = (5 * b) % (42 - size + 1)
        batches.append((at, [torch.empty(n, dtype=torch.float64, device="cuda")
                             for _ in range(size)],
                        [torch.empty_like(ins[at + k]) for k in range(size)]))

    def enqueue(at, spaces, outs):
        part = trs[at:at + len(spaces)]
        sp.multi_transform_backward(part, ins[at:at + len(spaces)], spaces)
        sp.multi_transform_forward(part, spaces, outs, [sp.SPFFT_FULL_SCALING] * len(part))

    print(f"batch plans: {dims}", flush=True)
    torch.cuda.synchronize()
    for b in batches:
        enqueue(*b)
    torch.cuda.synchronize()
    for at, spaces, outs in batches:
        for k in range(len(spaces)):
            want = plans[(at + k) % 3].backward(vals[at + k])
            got = spaces[k].cpu().numpy().view(np.complex128).reshape(dims[::-1])
            assert orc.rel_l2(got, want) <= 1e-12, (len(spaces), k)
            back = outs[k].cpu().numpy().view(np.complex128)
            assert orc.rel_l2(back, plans[(at + k) % 3].forward(want, True)) <= 1e-12
    first = [x.clone() for x in batches[0][1] + batches[0][2]]
    for x in batches[0][1] + batches[0][2]:
        x.zero_()
    torch.cuda.synchronize()
    enqueue(*batches[0])
    torch.cuda.synchronize()
    for x, y in zip(first, batches[0][1] + batches[0][2]):
        assert torch.equal(x, y)
