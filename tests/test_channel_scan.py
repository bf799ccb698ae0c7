"""The scans of an input position's channels for its largest magnitude issue their loads in rounds, sixteen per lane, and
without a branch: a lane's channels past the group's are read all the same and not used.  What they read instead has to
be a channel of the group: a lane with no channel of its own (fewer channels than lanes across them) once read the
channel of its own number, planes past the end of the tensor in the last image.  No device is touched."""
import os
import re
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
KERNELS = os.path.join(ROOT, "nnabla_amd", "csrc", "kernels")

PROGRAM = r"""
#include <cstddef>
#include "gemm_layout.hpp"
#include <cstdio>
int main() {
  for (int Cg = 1; Cg <= 600; ++Cg)
    for (int c = 0; c < Cg + 16 * 16 + 16; ++c) {
      const int at = nbla_hip::scan_channel(c, Cg);
      if (at < 0 || at >= Cg || (c < Cg && at != c)) {
        printf("%d of %d reads %d\n", c, Cg, at);
        return 1;
      }
    }
  return 0;
}
"""


def test_a_channel_past_the_groups_reads_one_of_the_groups(tmp_path):
    src, exe = tmp_path / "scan.cpp", tmp_path / "scan"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++14", "-D__host__=", "-D__device__=", "-I", KERNELS, "-o", str(exe), str(src)],
                   check=True)
    done = subprocess.run([str(exe)], capture_output=True, text=True)
    assert done.returncode == 0, done.stdout


def test_every_scan_takes_its_channels_from_it():
    scans = 0
    for name in ("gemm_bits.hip", "conv.hip"):
        text = open(os.path.join(KERNELS, name)).read()
        # the loads of a round: plane `index` of the position's image
        indices = re.findall(r"v(?:\[slot\])?\[j\] = src\[\(int64_t\)(.+?) \* plane\];", text)
        assert indices and set(indices) == {"scan_channel(c, Cg)"}, (name, indices)
        scans += len(indices)
    assert scans == 3
