"""GPU: edus_lindhard_device_noalloc, the entry point for code under graph
capture, runs the same kernels there as everywhere: its first call in a process
that needs more than 64 KB of LDS (8 bands, 3 filled, 48 x 48) is captured, and
every replay, with the program's own work between, equals
edus_lindhard_device's result bit for bit.  In a process of its own, so that no
other test has made that first call."""
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = """
import sys
sys.path[:0] = [%r, %r]
import numpy as np, torch, edus
import screened_models as sm

def arrays(nb, n, seed):
    U, w = sm.random_bands(nb, n, n, seed=seed)
    X = torch.zeros((nb * nb, n * n), dtype=torch.complex128, device="cuda")
    return torch.from_numpy(U).cuda(), torch.from_numpy(np.ascontiguousarray(w)).cuda(), X

def call(nb, nf, n, a, stream):
    edus.lindhard_device_noalloc(nb, n, n, nf, a[0].data_ptr(), a[1].data_ptr(), a[2].data_ptr(), stream)

small, big = arrays(2, 6, 1), arrays(8, 48, 2)
call(2, 1, 6, small, torch.cuda.current_stream().cuda_stream)  # the library and its scratch are there
torch.cuda.synchronize()
graph = torch.cuda.CUDAGraph()
with torch.cuda.graph(graph):
    call(8, 3, 48, big, torch.cuda.current_stream().cuda_stream)
work, ref = torch.empty_like(big[0]), torch.empty_like(big[2])
for r in range(3):
    big[2].zero_()
    graph.replay()
    torch.cuda.synchronize()
    edus.lindhard_device(8, 48, 48, 3, big[0].data_ptr(), big[1].data_ptr(), work.data_ptr(), ref.data_ptr(),
                         torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    assert ref.abs().max().item() > 0 and torch.equal(big[2], ref), r
print("equal")
""" % (os.path.join(ROOT, "edus_2.0_amd"), os.path.join(ROOT, "tests"))


def test_first_call_under_capture():
    r = subprocess.run([sys.executable, "-c", PROGRAM], capture_output=True, text=True, timeout=100)
    print(r.stdout, r.stderr[-2000:], flush=True)
    assert r.returncode == 0 and "equal" in r.stdout
