"""The hand-over of an LDS slot in csrc/gemm_ring.hpp, seen in the assembly that the compiler makes of it."""
import os
import re
import subprocess

import pytest

from dejavu_amd.build import CSRC, HIPCC_FLAGS, hipcc_path

SOURCE = """
#include "gemm_ring.hpp"
struct Store {
  float* y;
  int ldy;
  __device__ void operator()(int m, int n, dv::float4_t v) const { *reinterpret_cast<dv::float4_t*>(y + (long)n * ldy + m) = v; }
};
#define RING(MB, NB, KC, ST, WM, WN) \\
  template __global__ void dv::gemm_ring_kernel<dv::half_t, MB, NB, KC, ST, WM, WN, false>( \\
      dv::RingOperands<dv::half_t>, dv::PlainRows, Store, dv::float4_t*);
RING(32, 16, 128, 4, 2, 1)
RING(64, 64, 64, 4, 2, 2)
RING(192, 192, 64, 3, 2, 4)
"""


def test_reads_have_returned_before_a_slot_is_loaded_again(tmp_path):
    """Behind the barrier the slot that was read last is loaded again, by other waves too: each wave's own reads and its part
    of the next slot are waited for in front of it."""
    try:
        hipcc = hipcc_path()
    except RuntimeError as e:
        pytest.skip(str(e))
    src, out = tmp_path / "ring.hip", tmp_path / "ring.s"
    src.write_text(SOURCE)
    flags = [f for f in HIPCC_FLAGS if f not in ("-shared", "-fPIC")]
    subprocess.run([hipcc, *flags, "-w", "-S", "--cuda-device-only", "-I", CSRC, "-I", os.path.join(CSRC, "..", "..", "include"),
                    str(src), "-o", str(out)], check=True)
    lines = [line.split(";")[0].strip() for line in out.read_text().splitlines()]
    barriers = [i for i, line in enumerate(lines) if line.startswith("s_barrier")]
    assert len(barriers) >= 3
    for i in barriers:
        before = []
        for line in reversed(lines[:i]):
            if line.endswith(":") or line.startswith(("ds_read", "buffer_load", "global_load", "s_cbranch")):
                break
            before.append(line)
        waits = " ".join(line for line in before if line.startswith("s_waitcnt"))
        assert re.search(r"lgkmcnt\(0\)", waits) and re.search(r"vmcnt\(\d+\)", waits), before


def test_sums_of_the_narrowest_tile_are_waited_for(tmp_path):
    """One matrix instruction a step leaves nothing between the last of them and the reads of its sums: the wait stands in the
    kernel, in front of the branch that leaves the loop."""
    try:
        hipcc = hipcc_path()
    except RuntimeError as e:
        pytest.skip(str(e))
    src, out = tmp_path / "ring.hip", tmp_path / "ring.s"
    src.write_text("\n".join(SOURCE.splitlines()[:-2]))
    flags = [f for f in HIPCC_FLAGS if f not in ("-shared", "-fPIC")]
    subprocess.run([hipcc, *flags, "-w", "-S", "--cuda-device-only", "-I", CSRC, "-I", os.path.join(CSRC, "..", "..", "include"),
                    str(src), "-o", str(out)], check=True)
    lines = [line.split(";")[0].strip() for line in out.read_text().splitlines()]
    lines = lines[next(i for i, line in enumerate(lines) if re.match(r"_ZN2dv16gemm_ring.*Li32ELi16E.*:$", line)):]
    last = max(i for i, line in enumerate(lines) if line.startswith("v_mfma"))
    behind = lines[last + 1:next(i for i in range(last + 1, len(lines)) if lines[i].startswith(("s_cbranch", "s_branch")))]
    assert "s_nop 7" in behind, behind
