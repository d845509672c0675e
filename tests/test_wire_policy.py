"""Which decodes of the FP8 wire store non-temporally (xgen_amd/csrc/wire_policy.h, the same source text
the launch compiles), on the host with g++."""
import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]

CHECK = r"""
#include <cstdio>
#include <cstdlib>
#include "wire_policy.h"
int main(int argc, char **argv) {
  for (int i = 1; i + 4 < argc; i += 5)
    printf("%d ", (int)xgen::decode_stores_non_temporal(atoll(argv[i]), 256ll << 20, atoll(argv[i + 1]), atoi(argv[i + 2]),
                                                        atoi(argv[i + 3]) != 0, strtoull(argv[i + 4], nullptr, 10)));
}
"""

MB = 1 << 20
# (bytes of the call, bytes of an output row, lanes per row, strided, base and stride bits) -> non-temporal
CASES = [
    ((256 * MB, 256, 8, 0, 0), 0),       # the last call that the cache holds
    ((256 * MB + 1, 256, 8, 0, 0), 1),
    ((900 * MB, 256, 8, 0, 4096), 1),    # whole lines, contiguous: no upper line
    ((384 * MB, 256, 8, 1, 768), 1),     # strided, whole 64-byte pieces: up to 1.5 caches
    ((384 * MB + 1, 256, 8, 1, 768), 0),
    ((384 * MB, 128, 4, 0, 0), 1),       # rows of 64 values: 64 bytes a store
    ((450 * MB, 128, 4, 0, 0), 0),
    ((450 * MB, 192, 8, 0, 0), 0),       # rows of 96 values end in half a line
    ((300 * MB, 256, 8, 0, 64), 1),      # a base 64 bytes off a line
    ((450 * MB, 256, 8, 0, 64), 0),
    ((300 * MB, 256, 8, 0, 16), 0),      # pieces that no store instruction fills: never
    ((300 * MB, 256, 8, 1, 96), 0),
    ((300 * MB, 16, 1, 0, 0), 0),
    ((300 * MB, 64, 2, 0, 0), 0),
    ((300 * MB, 80, 4, 0, 0), 0),
    ((300 * MB, 272, 16, 0, 0), 0),
]


def test_non_temporal_decodes(tmp_path):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("g++ not available")
    src, exe = tmp_path / "check.cpp", tmp_path / "check"
    src.write_text(CHECK)
    subprocess.run([gxx, "-O1", "-std=c++17", f"-I{ROOT / 'xgen_amd' / 'csrc'}", str(src), "-o", str(exe)], check=True)
    args = [str(v) for case, _ in CASES for v in case]
    out = subprocess.run([str(exe), *args], stdout=subprocess.PIPE, text=True, check=True, timeout=60).stdout
    assert [int(v) for v in out.split()] == [want for _, want in CASES]
