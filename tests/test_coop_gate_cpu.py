"""Which errors of a cooperative launch mean that none are to be had, and how
long the traversals wait before they ask again: the rule alone, compiled for the
host."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include "graph.hpp"

int main() {
  using mgg::CoopGate;
  const hipError_t refusals[] = {hipErrorIllegalState, hipErrorNotSupported,
                                 hipErrorCooperativeLaunchTooLarge};
  const hipError_t errors[] = {hipErrorInvalidValue, hipErrorInvalidConfiguration,
                               hipErrorIllegalAddress, hipErrorLaunchFailure, hipErrorOutOfMemory,
                               hipErrorUnknown, hipErrorInvalidDeviceFunction};
  for (hipError_t e : errors) {
    CoopGate g;
    if (g.refused(e)) return 1;  // an error, not a refusal
    if (!g.open()) return 2;     // and nothing to remember
  }
  for (hipError_t e : refusals) {
    CoopGate g;
    for (int round = 0; round < 3; round++) {
      if (!g.open()) return 3;
      if (!g.refused(e)) return 4;
      for (int i = 0; i < CoopGate::WAIT; i++)
        if (g.open()) return 5;  // the next traversals take their other path
      if (!g.open()) return 6;   // then it is asked again, and open for good
      if (!g.open()) return 7;
    }
  }
  return 0;
}
"""


def test_refusals_and_errors(tmp_path):
    src, exe = tmp_path / "gate.cpp", tmp_path / "gate"
    src.write_text(PROGRAM)
    subprocess.check_call(["g++", "-std=c++17", "-O1", "-D__HIP_PLATFORM_AMD__",
                           "-I/opt/rocm/include",
                           "-I" + os.path.join(ROOT, "grus_framework_amd", "csrc"),
                           str(src), "-o", str(exe)])
    assert subprocess.run([str(exe)]).returncode == 0
