"""The room that crews take in a dense brick's stage, for the shipped layout and
for overrides of its size: the compiler checks the constants of vlj_device.h."""
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "virial-engine_amd", "csrc")
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"

CHECK = """
#include <hip/hip_runtime.h>
#include "vlj_device.h"
using namespace vlj;
// where wave w leaves its octet (an index into one of the three arrays) lies past
// every atom that a brick with crews stages, and ends before the sentinel
constexpr bool octets_fit() {
  for (long w = 0; w < (long)kCrewWaves; w++) {
    const long first = (long)Dense::kListPad - (w / 3 + 1) * (long)kCrewOctet;
    if (kCrewStaged > 0u && (first < (long)kCrewStaged || first + (long)kCrewOctet > (long)Dense::kListPad)) return false;
  }
  return kCrewStaged < Dense::kListPad;
}
static_assert(octets_fit(), "crews past the stage");
static_assert((kCrewStaged > 0u) == EXPECTED, "crews where there is room");
"""


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="needs hipcc")
@pytest.mark.parametrize("stage,threads,room", [
    (3200, 512, True),
    (1600, 512, True),
    (1536, 512, False),
    (1024, 512, False),
    (3200, 1024, True),
    (2048, 1024, False),
    (3200, 256, True),
])
def test_crews_stay_inside_the_stage(tmp_path, stage, threads, room):
    src = tmp_path / "room.hip"
    src.write_text(CHECK)
    r = subprocess.run([HIPCC, "--offload-arch=gfx950", "--offload-host-only", "-std=c++17", "-fsyntax-only",
                        f"-DVLJ_STAGE_MAX={stage}", f"-DVLJ_BRICK_THREADS={threads}",
                        f"-DEXPECTED={'true' if room else 'false'}", "-I", CSRC, str(src)],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
