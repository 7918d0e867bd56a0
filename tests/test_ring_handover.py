"""What csrc/gemm_ring.hpp relies on, seen in the assembly that the compiler makes of every form in which ``gemm_ring`` launches it:
the hand-over of an LDS slot, and the sums of the matrix instructions, which nothing in the hardware waits for."""
import os
import re
import subprocess

import pytest

from dejavu_amd.build import CSRC, HIPCC_FLAGS, hipcc_path

# Rows whose weight is read past the caches, and rows that stay in them; all tiles, as the rule launches them.
SOURCE = """
#include "gemm_ring.hpp"
struct Store {
  float* y;
  int ldy;
  __device__ void operator()(int m, int n, dv::float4_t v) const { *reinterpret_cast<dv::float4_t*>(y + (long)n * ldy + m) = v; }
};
struct KeptRows : dv::PlainRows {
  static constexpr bool kPastCaches = false;
};
struct Launch {
  template <auto KERNEL, typename... A>
  int operator()(dim3 grid, dim3 threads, size_t lds, hipStream_t s, A... args) const {
    hipLaunchKernelGGL(KERNEL, grid, threads, lds, s, args...);
    return 0;
  }
};
int all(const dv::RingPlan& p, const dv::RingOperands<dv::half_t>& a, Store out) {
  return dv::gemm_ring(p, a, dv::PlainRows{}, out, nullptr, nullptr, Launch{}) + dv::gemm_ring(p, a, KeptRows{}, out, nullptr, nullptr, Launch{});
}
"""
# States between a matrix instruction of eight passes and the first use of its sums by another kind
STATES = 8


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    """Name -> lines of every instance of gemm_ring_kernel."""
    try:
        hipcc = hipcc_path()
    except RuntimeError as e:
        pytest.skip(str(e))
    where = tmp_path_factory.mktemp("ring")
    src, out = where / "ring.hip", where / "ring.s"
    src.write_text(SOURCE)
    flags = [f for f in HIPCC_FLAGS if f not in ("-shared", "-fPIC")]
    subprocess.run([hipcc, *flags, "-w", "-S", "--cuda-device-only", "-I", CSRC, "-I", os.path.join(CSRC, "..", "..", "include"),
                    str(src), "-o", str(out)], check=True)
    found, name = {}, None
    for line in out.read_text().splitlines():
        line = line.split(";")[0].strip()
        if re.match(r"_ZN2dv16gemm_ring_kernel.*:$", line):
            name = line[:-1]
            found[name] = []
        elif line.startswith(".Lfunc_end"):
            name = None
        elif name and line and (not line.startswith(".") or line.endswith(":")):
            found[name].append(line)
    return found


def form(name):
    """(rows of W, rows of X, weight past the caches, begins at different columns)"""
    m = re.search(r"KernelI\w*?Li(\d+)ELi(\d+)E(?:Li\d+E){4}Lb(\d)E", name.replace("_kernel", "Kernel"))
    return int(m[1]), int(m[2]), m[3] == "1", name.count("Lb1E") - (m[3] == "1") == 1


def test_every_form_is_here(kernels):
    forms = {form(name) for name in kernels}
    assert {f for f in forms if f[:2] == (32, 16)} == {(32, 16, True, False), (32, 16, True, True)}
    assert {f[:2] for f in forms} == {(32, 16), (64, 32), (128, 32), (64, 64), (96, 64), (128, 64), (64, 128), (128, 128), (192, 128), (64, 192),
                                      (128, 192), (192, 192), (64, 256), (128, 256)}


def test_reads_have_returned_before_a_slot_is_loaded_again(kernels):
    """Behind the barrier the slot that was read last is loaded again, by other waves too: each wave's own reads and its part
    of the next slot are waited for in front of it."""
    for name, lines in kernels.items():
        barriers = [i for i, line in enumerate(lines) if line.startswith("s_barrier")]
        assert barriers, name
        for i in barriers:
            before = []
            for line in reversed(lines[:i]):
                if line.endswith(":") or line.startswith(("ds_read", "buffer_load", "global_load", "s_cbranch")):
                    break
                before.append(line)
            waits = " ".join(line for line in before if line.startswith("s_waitcnt"))
            assert re.search(r"lgkmcnt\(0\)", waits) and re.search(r"vmcnt\(\d+\)", waits), (name, before)


def registers(text):
    found = set()
    for kind, first, last in re.findall(r"\b([av])\[(\d+):(\d+)\]", text):
        found |= {kind + str(i) for i in range(int(first), int(last) + 1)}
    return found | {kind + n for kind, n in re.findall(r"\b([av])(\d+)\b", text)}


def states_before_use(lines, start, limit=1000):
    """The fewest states, over all ways from the matrix instruction at ``start``, before another kind of instruction reads its sums
    or a matrix instruction takes them as an operand; None if none does within ``limit``."""
    labels = {line[:-1]: i for i, line in enumerate(lines) if line.endswith(":")}
    sums, least, seen, ways = registers(lines[start].split(None, 1)[1].split(",")[0]), None, {}, [(start + 1, 0)]
    while ways:
        at, states = ways.pop()
        while at < len(lines) and states < limit and seen.get(at, limit) > states:
            seen[at] = states
            op, _, rest = lines[at].partition(" ")
            at += 1
            if op.endswith(":"):
                continue
            if op == "s_endpgm":
                break
            if op.startswith(("s_branch", "s_cbranch")):
                ways.append((labels[rest.strip()], states + 1))
                if op == "s_branch":
                    break
            elif op.startswith(("v_", "ds_", "global_", "buffer_", "flat_")):
                operands = re.findall(r"[av]\[\d+:\d+\]|\b[av]\d+\b", rest)
                matrix, stores = op.startswith("v_mfma"), "store" in op or "write" in op or "lds" in op
                read = operands if stores else operands[1:3] if matrix else operands[1:]
                if sums & set().union(*map(registers, read)):
                    least = states if least is None else min(least, states)
                    break
                if operands and not stores and registers(operands[0]) & sums:  # added to or written over
                    break
            states += int(rest) + 1 if op == "s_nop" else 1
    return least


def test_sums_are_waited_for(kernels):
    """All ways out of all loops of all forms.  (One matrix instruction a step, as in the narrowest tile, leaves nothing between the
    last of them and the reads of its sums: there the wait stands in the kernel.)"""
    for name, lines in kernels.items():
        uses = [states_before_use(lines, i) for i, line in enumerate(lines) if line.startswith("v_mfma_f32_16x16x32")]
        uses = [u for u in uses if u is not None]
        assert uses and min(uses) >= STATES, (name, sorted(uses)[:4])


def test_too_few_states_are_seen():
    step = ["v_mfma_f32_16x16x32_f16 v[0:3], v[4:7], v[8:11], v[0:3]", "s_cbranch_scc1 .LBB0_1"]
    assert states_before_use(step + ["s_nop 7", ".LBB0_1:", "v_add_f32_e32 v20, v3, v4"], 0) == 1
    assert states_before_use(step + [".LBB0_1:", "s_nop 7", "s_nop 1", "v_add_f32_e32 v20, v3, v4"], 0) == 11
    assert states_before_use([step[0], "global_store_dwordx4 v[20:21], v[0:3], off"], 0) == 0
    assert states_before_use([step[0], "v_mov_b32_e32 v0, v9", "s_endpgm"], 0) is None
