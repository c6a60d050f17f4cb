"""Kernel attributes are set on every device that a process uses (CPU only:
the header is compiled for the host with a stand-in for the runtime call)."""
import glob
import os
import re
import subprocess

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                    "pylabolt_amd", "csrc")

PROGRAM = r"""
#include "d2q9_per_device.h"
#include <cstdio>
#include <initializer_list>
int main() {
  d2q9::PerDevice a, b;
  int calls[70] = {}, fail = 0;
  auto set = [&](d2q9::PerDevice& p, int dev) {
    return p.once(dev, [&] { ++calls[dev]; return fail; });
  };
  fail = 7;
  std::printf("%d ", set(a, 1));            // fails, and is not remembered
  fail = 0;
  for (int n = 0; n < 3; ++n)
    for (int dev : {0, 1, 63, 65}) set(a, dev);
  set(b, 0);                                // another kernel's
  std::printf("%d %d %d %d\n", calls[0], calls[1], calls[63], calls[65]);
}
"""


def test_once_for_every_device(tmp_path):
    src = tmp_path / "p.cpp"
    src.write_text(PROGRAM)
    exe = str(tmp_path / "p")
    subprocess.run(["g++", "-std=c++17", "-I", CSRC, str(src), "-o", exe],
                   check=True)
    out = subprocess.run([exe], check=True, capture_output=True, text=True)
    assert out.stdout.split() == ["7", "2", "2", "1", "3"]


def test_no_attribute_is_set_once_per_process():
    found = 0
    for path in glob.glob(os.path.join(CSRC, "d2q9_*")):
        with open(path) as fh:
            text = fh.read()
        assert not re.search(r"static\s+const\s+hipError_t", text), path
        found += text.count("hipFuncSetAttribute(")
    assert found == 1       # allow_lds, through PerDevice
