"""How a digit x digit product's contraction is split over blocks (csrc/kernels/gemm_layout.hpp), compiled for the host: every
filled k tile belongs to one split, no split is empty, the splits fit the scratch that they were given, and leaving out the
tiles that are only padding never makes a split longer than it was with them (sixteen splits of 16 tiles once became eleven
of 24 that way).  No device is touched."""
import os
import subprocess

KERNELS = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "nnabla_amd", "csrc", "kernels")

PROGRAM = r"""
#include <cstddef>
#include "gemm_layout.hpp"
#include <cstdio>
#include <initializer_list>
using namespace nbla_hip;
int main() {
  const int64_t counts[] = {1, 2, 3, 5, 8, 15, 16, 17, 31, 64, 100, 128, 129, 256, 1000};
  for (int64_t K = 1; K <= kChunkK; ++K) {
    const int64_t padded = digit_k_tiles(K), filled = ceil_div(ceil_div(K, kTileK), 4) * 4;
    for (int64_t tiles : counts)
      for (int64_t most : {int64_t(0), int64_t(1), int64_t(2), int64_t(7), int64_t(1) << 40}) {
        const DigitSplit s = digit_split(tiles, padded, filled, most), whole = digit_split(tiles, padded, padded, most);
        const bool covers = s.count * s.tiles >= filled && (s.count - 1) * s.tiles < filled;
        if (!covers || s.tiles % 8 != 0 || (s.count > 1 && s.count > most) || s.tiles > whole.tiles ||
            (s.count > 1 && s.count * tiles > 256)) {
          printf("K %d, %d tiles, at most %d: %d of %d\n", (int)K, (int)tiles, (int)most, (int)s.count, (int)s.tiles);
          return 1;
        }
      }
  }
  const DigitSplit s = digit_split(1, digit_k_tiles(8032), 252, 1 << 20);
  printf("%d %d\n", (int)s.count, (int)s.tiles);
  return 0;
}
"""


def test_splits(tmp_path):
    src, exe = tmp_path / "split.cpp", tmp_path / "split"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++14", "-O1", "-D__host__=", "-D__device__=", "-I", KERNELS, "-o", str(exe), str(src)],
                   check=True)
    done = subprocess.run([str(exe)], capture_output=True, text=True)
    assert done.returncode == 0 and done.stdout.split() == ["16", "16"], done.stdout


def test_the_product_takes_its_splits_from_there():
    text = open(os.path.join(KERNELS, "gemm_digits.hip")).read()
    assert "digit_split(blocks, padded_tiles, chunk_tiles, most)" in text and "part.split_tiles = split.tiles;" in text
