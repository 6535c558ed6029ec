"""Creating an operator when device memory runs out: tables and inboxes that
only a faster form needs may be missing (the operator then takes the form that
does without), everything else fails the call.  On the CPU: the library's calls
of the HIP memory functions go to host memory, of which one allocation is
refused."""

import os
import subprocess
import sys

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

STUB = r"""
#include <stdlib.h>
#include <string.h>
static int calls, refused = -1;
void stub_refuse(int n) { calls = 0; refused = n; }
int stub_calls(void) { return calls; }
int hipMalloc(void **p, size_t n)
{
  *p = 0;
  if (calls++ == refused)
    return 2;
  *p = malloc(n);
  return 0;
}
int hipFree(void *p) { free(p); return 0; }
int hipMemcpy(void *d, const void *s, size_t n, int k)
{ (void)k; memcpy(d, s, n); return 0; }
int hipMemset(void *d, int v, size_t n) { memset(d, v, n); return 0; }
int hipStreamSynchronize(void *s) { (void)s; return 0; }
int hipGetLastError(void) { return 0; }
"""

SCRIPT = r"""
import ctypes, sys
stub = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
import hyperdeal_amd as H

def outcomes(make):
    stub.stub_refuse(-1)
    keep = make()
    total, out = stub.stub_calls(), []
    del keep
    for n in range(total):
        stub.stub_refuse(n)
        try:
            keep = make()
            del keep
            out.append(1)
        except H.HyperdealError:
            out.append(0)
    return out

mf = H.MatrixFree(2, 2, 2, [3, 2, 2, 3], [-1.0] * 4, [1.0] * 4)
mf.set_deformation(0.1, 2)
print(outcomes(lambda: H.AdvectionOperation(mf, [1.0, 0.5, -0.3, 0.2])))
mv = H.MatrixFree(2, 2, 3, [4, 4, 2, 2], [-1.0] * 4, [1.0] * 4)
print(outcomes(lambda: H.VlasovPoissonOperation(mv)))
"""


def test_optional_allocations(tmp_path):
    src, lib = tmp_path / "stub.c", tmp_path / "stub.so"
    src.write_text(STUB)
    subprocess.run(["gcc", "-shared", "-fPIC", "-o", str(lib), str(src)],
                   check=True)
    r = subprocess.run([sys.executable, "-c", SCRIPT, str(lib)], cwd=ROOT,
                       capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stderr
    curved, vp = [eval(line) for line in r.stdout.split("\n")[:2]]
    # the geometry's table, then two spaces' tables in both precisions and
    # their masks
    assert curved == [0] + 6 * [1]
    # the strips' inboxes
    assert sum(vp) == 1 and len(vp) >= 8
