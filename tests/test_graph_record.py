"""Recording launches as graph nodes: a node that cannot be added fails the recording, whatever
the runtime's last error says.  A host program over the library's own source, with the runtime's
call that adds a node replaced; no GPU."""
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "abd-warp_amd", "csrc")
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"

PROGRAM = r"""
#include <hip/hip_runtime.h>
#include <cstdio>
#include "abd_internal.h"

static int calls = 0, fail_at = 0;
extern "C" hipError_t hipGraphAddKernelNode(hipGraphNode_t* node, hipGraph_t, const hipGraphNode_t* deps,
                                            size_t n, const hipKernelNodeParams*) {
    if (++calls == fail_at) return hipErrorOutOfMemory;
    if ((n == 0) != (calls == 1) || (n && *deps != (hipGraphNode_t)(size_t)(calls - 1))) return hipErrorUnknown;
    *node = (hipGraphNode_t)(size_t)calls;
    return hipSuccess;
}
extern "C" hipError_t hipGetLastError() { return hipSuccess; }

static void kernel(int, double) {}

static int record(int launches, int fail) {
    calls = 0;
    fail_at = fail;
    abd::graph_record((hipGraph_t)1);
    for (int k = 0; k < launches; ++k) abd::launch_kernel(kernel, dim3(1), dim3(64), 0, (hipStream_t)0, k, 0.5);
    const int rc = abd::graph_record_end();
    if (abd::capturing()) return 1;
    return rc;
}

int main() {
    const int want = -(int)hipErrorOutOfMemory;
    const int whole = record(3, 0), n = calls;
    const int first = record(3, 1), n1 = calls;
    const int last = record(3, 3), n2 = calls;
    const int after = record(2, 0);
    std::printf("%d %d %d %d, %d %d %d\n", whole, first == want, last == want, after, n, n1, n2);
    return 0;
}
"""


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="no hipcc")
def test_a_node_that_cannot_be_added_fails_the_recording(tmp_path):
    src, exe = tmp_path / "record.cpp", tmp_path / "record"
    src.write_text(PROGRAM)
    subprocess.run([HIPCC, "-x", "hip", "--offload-arch=gfx950", "-O1", "-std=c++17", "-I", CSRC, str(src),
                    os.path.join(CSRC, "abd_common.hip"), "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
                    "-w", "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], check=True, capture_output=True, text=True).stdout
    # nodes are added one after the other, and none after a failure
    assert out.strip() == "0 1 1 0, 3 1 3"
