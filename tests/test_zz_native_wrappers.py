"""The native wrappers beside other Python threads (MI355X only)."""

import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

# An allocator whose every allocation takes a while, as one that waits for the
# device does.
ALLOCATOR = r"""
#include <hip/hip_runtime_api.h>
#include <sys/types.h>
#include <time.h>
static int slow = 0;
extern "C" void make_slow(int on) { slow = on; }
extern "C" void* slow_alloc(ssize_t size, int device, hipStream_t stream) {
  if (slow) {
    struct timespec t = {0, 200000000};
    nanosleep(&t, 0);
  }
  void* p = 0;
  if (hipMalloc(&p, size > 0 ? size : 1) != hipSuccess) return 0;
  return p;
}
extern "C" void slow_free(void* p, ssize_t size, int device, hipStream_t stream) { (void)hipFree(p); }
"""

# Counts how often another thread runs while the main one is in a call of two
# allocations of 0.2 s each: of the wrapper, and of torch itself.
CHILD = r"""
import ctypes, sys, threading, time
import torch
path = sys.argv[1]
alloc = torch.cuda.memory.CUDAPluggableAllocator(path, "slow_alloc", "slow_free")
torch.cuda.memory.change_current_allocator(alloc)
slow = ctypes.CDLL(path).make_slow
from quail_amd import kernels as K
x = torch.zeros(4, 512, dtype=torch.bfloat16, device="cuda")
w = torch.ones(512, dtype=torch.bfloat16, device="cuda")
K.add_rmsnorm_quant(x, w, 1e-6)
torch.cuda.synchronize()
ticks, stop = [0], threading.Event()
def other():
    while not stop.is_set():
        ticks[0] += 1
        time.sleep(0.005)
thread = threading.Thread(target=other)
thread.start()
slow(1)
for call in (lambda: [torch.empty_like(x) for _ in range(2)], lambda: K.add_rmsnorm_quant(x, w, 1e-6)):
    before, start = ticks[0], time.time()
    keep = call()
    print("TICKS", ticks[0] - before, "SECONDS", time.time() - start, flush=True)
slow(0)
stop.set()
thread.join()
"""


def test_an_allocation_does_not_stop_other_threads(tmp_path):
    """A wrapper whose allocations take 0.4 s lets another thread run meanwhile
    (at least half as often as its 5 ms sleeps allow), as torch's own do."""
    source, lib = tmp_path / "alloc.cpp", tmp_path / "alloc.so"
    source.write_text(ALLOCATOR)
    subprocess.run(["g++", "-O1", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__=1", "-I/opt/rocm/include",
                    str(source), "-o", str(lib), "-L/opt/rocm/lib", "-lamdhip64"], check=True,
                   timeout=60)
    out = subprocess.run([sys.executable, "-u", "-c", CHILD, str(lib)], capture_output=True, text=True,
                         timeout=100, cwd=ROOT)
    assert out.returncode == 0, out.stderr[-2000:]
    lines = [x.split() for x in out.stdout.splitlines() if x.startswith("TICKS")]
    assert len(lines) == 2, out.stdout
    for line in lines:
        assert float(line[3]) >= 0.4 and int(line[1]) >= 40, lines
