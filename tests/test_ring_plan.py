"""Which tiles csrc/gemm_ring.hpp plans, asked of its host code."""
import os
import subprocess

import pytest

from dejavu_amd.build import CSRC, hipcc_path

SOURCE = """
#include <cstdio>
#include "gemm_ring.hpp"
int main() {
  int n, M, K, units;
  while (scanf("%d %d %d %d", &n, &M, &K, &units) == 4) {
    const dv::RingPlan p = dv::plan_ring(n, M, K, units);
    printf("%d %d %d %d %d\\n", p.mb, p.nb, p.rows, p.cols, p.splits);
  }
}
"""
ROWS = (2, 16, 17, 32, 33, 64, 65, 96, 128, 129, 192, 193, 256, 257, 320, 384, 385, 512)
WEIGHTS = [(M, K) for M in (4, 96, 768, 2048, 4096, 5120, 9216, 12288, 14400, 16384, 22016, 36864, 50272)
           for K in (8, 264, 768, 2048, 4096, 5120, 12288, 20480)]


@pytest.fixture(scope="module")
def plan(tmp_path_factory):
    try:
        hipcc = hipcc_path()
    except RuntimeError as e:
        pytest.skip(str(e))
    at = tmp_path_factory.mktemp("plan")
    src, exe = at / "plan.hip", at / "plan"
    src.write_text(SOURCE)
    subprocess.run([hipcc, "--offload-arch=gfx950", "-std=c++17", "-w", "-I", CSRC, "-I", os.path.join(CSRC, "..", "..", "include"),
                    str(src), "-o", str(exe)], check=True)

    def ask(questions):
        out = subprocess.run([str(exe)], input="\n".join(" ".join(map(str, q)) for q in questions), text=True, check=True,
                             capture_output=True).stdout
        return [tuple(map(int, line.split())) for line in out.splitlines()]

    return ask


@pytest.mark.parametrize("units", [32, 64, 128, 256])
def test_splits_fill_the_compute_units_of_the_device_and_no_more(plan, units):
    """K is split only while the workgroups are no more than the device's round of them (four times that for 16 rows, an
    eighth more up to 64), whatever the number of its compute units; every tile and row is covered."""
    asked = [(n, M, K, units) for n in ROWS for M, K in WEIGHTS]
    for (n, M, K, _), (mb, nb, rows, cols, splits) in zip(asked, plan(asked)):
        assert rows * mb >= M > (rows - 1) * mb and cols * nb >= n > (cols - 1) * nb
        assert 1 <= splits <= min(8, max(1, K // 256))
        most = 4 * units if nb == 16 else units * 9 // 8 if nb <= 64 else units
        assert splits == 1 or splits * rows * cols <= most, (n, M, K, mb, nb, splits)


def test_a_quarter_of_the_compute_units_takes_a_quarter_of_the_rows(plan):
    """The lines of the rule that stand for a round of workgroups move with the device."""
    # 47 rows: the taller tile; 96 rows: 64 weight rows a tile up to one round of them
    asked = [(47, 16384, 4096, 256), (47, 4096, 4096, 64), (47, 4095, 4096, 64), (96, 16384, 2048, 256), (96, 16448, 2048, 256),
             (96, 8192, 2048, 128), (96, 8256, 2048, 128)]
    assert [p[0] for p in plan(asked)] == [96, 96, 64, 64, 128, 64, 128]


def test_small_weights_of_65_to_128_rows(plan):
    """Tiles of 64 weight rows from 4096 to below 6144 columns, where those of 128 would have an eighth of the columns each."""
    asked = [(n, 4096, K, 256) for n in (65, 128) for K in (4088, 4096, 6136, 6144, 8184)] + [(100, 4224, 4096, 256), (64, 4096, 4096, 256)]
    assert [p[0] for p in plan(asked)] == [128, 64, 64, 128, 128] * 2 + [128, 64]


def test_which_windows_multiply_live_rows_only(tmp_path):
    """Both sides of each line: rows of the window, size of a head, chosen heads."""
    try:
        hipcc = hipcc_path()
    except RuntimeError as e:
        pytest.skip(str(e))
    src, exe = tmp_path / "live.hip", tmp_path / "live"
    src.write_text('#include <cstdio>\n#include "../../include/dejavu_hip.h"\n#include "qkv_window.hpp"\nint main() { int t, n, hd, h; '
                   'while (scanf("%d %d %d %d", &t, &n, &hd, &h) == 4) printf("%d\\n", dv::window_live(t, n, hd, 3 * h * hd, 256)); }\n')
    subprocess.run([hipcc, "--offload-arch=gfx950", "-std=c++17", "-w", "-I", CSRC, "-I", os.path.join(CSRC, "..", "..", "include"),
                    str(src), "-o", str(exe)], check=True)
    asked = {(13, 16, 128, 24): 1, (12, 16, 128, 24): 0, (16, 12, 128, 24): 0, (16, 13, 128, 24): 1, (16, 5, 128, 96): 0, (9, 8, 128, 24): 0,
             (16, 32, 64, 48): 0, (16, 32, 32, 64): 0, (16, 32, 128, 10): 0, (16, 32, 128, 11): 1, (1, 32, 128, 24): 0}
    out = subprocess.run([str(exe)], input="\n".join("%d %d %d %d" % q for q in asked), text=True, check=True, capture_output=True).stdout
    assert list(map(int, out.split())) == list(asked.values())
