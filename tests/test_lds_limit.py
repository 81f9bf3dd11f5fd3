"""csrc/lds_limit.hpp against a runtime of its own: what a kernel may have of LDS is asked for on every device by itself, once, and again where it
was refused."""
import os
import shutil
import subprocess

import pytest

from based_amd import build

PROGRAM = r"""
#include "lds_limit.hpp"
static int device, asked[100], refuse;
extern "C" hipError_t hipGetDevice(int* d) { return *d = device, hipSuccess; }
extern "C" hipError_t hipFuncSetAttribute(const void*, hipFuncAttribute, int) { return ++asked[device], refuse ? hipErrorInvalidValue : hipSuccess; }
int main() {
  static based::LdsAllowed one, other;
  const size_t large = 154 * 1024;
  int bad = based::allow_lds(&one, 64 * 1024, one) != hipSuccess || asked[0] != 0;  // (needs no leave)
  for (int i = 0; i < 3; ++i) bad |= based::allow_lds(&one, large, one) != hipSuccess || asked[0] != 1;
  device = 1, refuse = 1;
  bad |= based::allow_lds(&one, large, one) == hipSuccess || asked[1] != 1;
  refuse = 0;
  for (int i = 0; i < 3; ++i) bad |= based::allow_lds(&one, large, one) != hipSuccess || asked[1] != 2;
  bad |= based::allow_lds(&other, large, other) != hipSuccess || asked[1] != 3;
  device = 0;
  bad |= based::allow_lds(&one, large, one) != hipSuccess || asked[0] != 1;
  device = based::kMaxDevices;
  return bad | (based::allow_lds(&one, large, one) == hipSuccess);
}
"""


def test_every_device_is_asked(tmp_path):
    if shutil.which("g++") is None:
        pytest.skip("no host compiler")
    (tmp_path / "t.cpp").write_text(PROGRAM)
    rocm = os.path.dirname(os.path.dirname(os.path.realpath(build.HIPCC)))
    include = next(p for p in (os.path.join(rocm, "include"), "/opt/rocm/include") if os.path.exists(os.path.join(p, "hip", "hip_runtime_api.h")))
    subprocess.run(["g++", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-isystem", include, "-I", build.CSRC, str(tmp_path / "t.cpp"), "-o", str(tmp_path / "t")],
                   check=True)
    assert subprocess.run([str(tmp_path / "t")]).returncode == 0


@pytest.mark.parametrize("source", sorted(f for f in os.listdir(build.CSRC) if f.endswith(".hip")))
def test_no_kernel_is_allowed_once_for_a_process(source):
    """Whoever asks the runtime itself keeps the answer by device."""
    text = open(os.path.join(build.CSRC, source)).read()
    assert "hipFuncSetAttribute" not in text or "allowed[dev]" in text
