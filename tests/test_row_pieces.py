"""The shift that puts a 16-byte piece crossing the end of a row into place
(shift_piece, csrc/device_util.hpp), on the host.

The unaligned row loads read such a piece where the row ends and shift the
elements past the end out. The LayerNorm forward of a handle whose width is
not a multiple of 64 also asks for pieces wholly past the row's end (H's
padded columns), up to 63 columns past it, so the shift takes any count from
0 to 128 bits and beyond. The helper is compiled for the host with the
undefined-behaviour check of shifts, which ends the program at a count the
type does not have.
"""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "test-model-thing-cuda_amd", "csrc")
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")

pytestmark = pytest.mark.skipif(not os.path.exists(HIPCC) and shutil.which("hipcc") is None,
                                reason="hipcc not available")

PROGRAM = r"""
#include <cstdio>
#include "device_util.hpp"
int main() {
    const unsigned __int128 x = ((unsigned __int128)0xfedcba9876543210ull << 64) | 0x0123456789abcdefull;
    for (int bits = 0; bits <= 16 * (63 + 8); ++bits) {
        uint64_t lo = (uint64_t)x, hi = (uint64_t)(x >> 64);
        tmt::shift_piece(lo, hi, bits);
        const unsigned __int128 want = bits < 128 ? x >> bits : 0;
        if (lo != (uint64_t)want || hi != (uint64_t)(want >> 64)) {
            std::printf("wrong at %d bits\n", bits);
            return 1;
        }
    }
    std::printf("ok\n");
    return 0;
}
"""


def test_shift_piece_any_count(tmp_path):
    src, exe = tmp_path / "pieces.hip", tmp_path / "pieces"
    src.write_text(PROGRAM)
    r = subprocess.run([HIPCC, "--offload-host-only", "-std=c++17", "-O1", "-I", CSRC,
                        "-Xarch_host", "-fsanitize=shift", "-Xarch_host", "-fsanitize-trap=shift",
                        str(src), "-o", str(exe)], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stderr[-2000:]
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout == "ok\n", (r.returncode, r.stdout)
