"""CPU: the split of a KIVI tail over a workgroup's waves, for any number of them (BPT_DECODE_WAVES): every token of the
longest tail falls to exactly one round of one wave's 16-lane groups."""

import subprocess

import pytest

CHECK = """
#include "bpt_internal.h"
constexpr bool once(int waves) {
  int taken[4096] = {};
  for (int r = 0; r < bpt::kivi_tail_rounds(waves); ++r)
    for (int w = 0; w < waves; ++w)
      for (int lane = 0; lane < 64; lane += 16) ++taken[bpt::kivi_tail_token(waves, r, w, lane)];
  for (int t = 0; t < bpt::kKiviMaxTail; ++t)
    if (taken[t] != 1) return false;
  return true;
}
static_assert(once(WAVES), "a token is taken twice or not at all");
"""


@pytest.mark.parametrize("waves", [1, 2, 3, 4, 8, 16])
def test_every_tail_token_falls_to_one_wave(waves, tmp_path):
    from bpt_amd import _build

    src = tmp_path / "check.hip"
    src.write_text(CHECK)
    cmd = [_build.hipcc(), "-std=c++17", "--cuda-host-only", "-fsyntax-only", f"-DWAVES={waves}", f"-I{_build.CSRC}", str(src)]
    proc = subprocess.run(cmd, capture_output=True, text=True)
    assert proc.returncode == 0, proc.stderr[-2000:]


@pytest.mark.parametrize("waves", [2, 8])
def test_the_kernel_compiles_with_other_wave_counts(waves):
    from bpt_amd import _build

    cmd = [_build.hipcc(), f"--offload-arch={_build.ARCH}", "-std=c++17", "--cuda-device-only", "-fsyntax-only",
           f"-DBPT_DECODE_WAVES={waves}", f"-I{_build.INCLUDE}", f"-I{_build.CSRC}", str(_build.CSRC / "kivi_decode.hip")]
    proc = subprocess.run(cmd, capture_output=True, text=True)
    assert proc.returncode == 0, proc.stderr[-2000:]
