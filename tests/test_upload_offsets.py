"""Offsets below 0 are refused like any that step back, by the check kernels and
by the host's restatement, without a look at the slot before the first one."""
import numpy as np
import pytest

from oracle import prep
from helpers import random_graph


def refused(side, value):
    from everest_amd import abi
    rng = np.random.default_rng(9)
    U, V, T = random_graph(rng, 300, 30, 1000)
    U[0], V[0], T[0] = 40, 41, -1   # vertex 0 has one out-edge, vertex 1 one in-edge
    g = {k: np.array(v) if isinstance(v, np.ndarray) else v for k, v in prep.preprocess(U, V, T).items()}
    x = 1 if side == "out" else 2   # an offset whose list begins with slot 0 once the ones before are empty
    R, P = g[side + "R"], g[side + "V"]
    if side == "out":               # the first slot's edge is another vertex's
        P[0], P[1] = P[1], P[0]
    R[x] = value
    with pytest.raises(abi.TMError) as e:
        abi.DeviceGraph.from_dict(g)
    assert e.value.status == 1
    return str(e.value)


@pytest.mark.parametrize("side", ["out", "in"])
@pytest.mark.parametrize("value", [-1, -5, -2**31])
def test_refused_without_gpu(side, value):
    from everest_amd import abi
    if abi.lib().tm_device_count() > 0:
        pytest.skip("the check kernels run here")
    assert "CSR" in refused(side, value)


@pytest.mark.gpu
@pytest.mark.parametrize("side", ["out", "in"])
@pytest.mark.parametrize("value", [-1, -5, -2**31])
def test_refused_on_gpu(side, value):
    print(side, value, flush=True)
    assert "CSR offsets not monotone" in refused(side, value)


HARNESS = """
#include <algorithm>
#include <sys/mman.h>
#include "tm_types.h"
using std::max;
#define __global__
#define __launch_bounds__(n)
#define __restrict__
struct { int x; } blockIdx, blockDim = {256}, threadIdx;
static void atomicOr(unsigned *p, unsigned v) { *p |= v; }
enum { V_CSR = 8 };
constexpr int V_CSR_SIDE = 5;
%s
int main() {
  // vertex 0 without edges, slots 0 and 1 vertex 1's; its offset below 0
  const int E = 2, V = 3;
  const tm_edge Eg[E] = {{1, 2, 0}, {1, 2, 1}};
  char *page = (char *)mmap(0, 8192, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS, -1, 0);
  int *P = (int *)(page + 4096);  // nothing may be read before it
  P[1] = 1;
  mprotect(page, 4096, PROT_NONE);
  const int R[V + 1] = {0, -3, 2, 2};
  unsigned bad = 0;
  for (threadIdx.x = 0; threadIdx.x < 256; threadIdx.x++) check_slots_kernel(Eg, R, P, E, V, 0, &bad);
  return bad != 0;
}
"""


def test_the_slots_check_reads_no_slot_before_the_first(tmp_path):
    """The kernel's own text on the host, the page before its list closed."""
    import os
    import re
    import subprocess
    src = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "everest_amd", "csrc", "hip")
    text = open(os.path.join(src, "tm_abi.hip")).read()
    kernel = re.search(r"__global__ void __launch_bounds__\(256\) check_slots_kernel\(.*?\n}\n", text, re.S).group(0)
    cc = tmp_path / "slots.cc"
    cc.write_text(HARNESS % kernel)
    exe = str(tmp_path / "slots")
    subprocess.check_call(["g++", "-std=c++17", "-g", "-I" + src, str(cc), "-o", exe])
    p = subprocess.run([exe], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    assert p.returncode == 0, p.stdout[:2000]
