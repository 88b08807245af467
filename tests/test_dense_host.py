"""Index arithmetic of the dense kernels that the host compiles too, at sizes no test can run."""
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "qwen3.ink.cpp_amd", "csrc")

# Against the place written out in 64 bits: around the last place of a sequence, around 2^24 places and around 2^32 entries of the tables.
ANGLES = r"""
#include <algorithm>
#include <cstdio>
#include "dense.h"
int main() {
    const int seqs[] = {1, 2, 33, 4352, (1 << 24) - 1, 1 << 24, (1 << 24) + 40, 150000000, 2147483647}, pairs[] = {1, 31, 32, 64, 2048};
    long long bad = 0, seen = 0;
    for (int seq : seqs)
        for (int p : pairs)
            for (long long pos : {0LL, 1LL, 500LL, (1LL << 24) - 16, 1LL << 24, 140000000LL, seq - 40LL, seq - 28LL, seq - 1LL})
                for (int m : {0, 4, 28, 4092}) {
                    if (pos < 0 || pos >= seq) continue;
                    const a81w41::AngleRows a((int)pos, m, seq, p);
                    for (int d = 0; d < 28; d++, seen++)
                        bad += a.base + a.behind(d) != (unsigned long long)std::min(pos + m + d, seq - 1LL) * p;
                }
    if (bad) printf("%lld of %lld\n", bad, seen);
    return bad || seen < 10000;
}
"""


@pytest.mark.skipif(not shutil.which("g++"), reason="no host compiler")
def test_angle_rows_of_long_sequences(tmp_path):
    source, exe = tmp_path / "angles.cpp", tmp_path / "angles"
    source.write_text(ANGLES)
    # the element type is not used here; g++ of this age has no __bf16
    built = subprocess.run(["g++", "-std=c++17", "-w", "-D__HIP_PLATFORM_AMD__", "-D__bf16=short", "-I/opt/rocm/include", "-I", CSRC, str(source),
                            "-o", str(exe)], capture_output=True, text=True)
    assert built.returncode == 0, built.stderr[-2000:]
    run = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert run.returncode == 0, run.stdout
