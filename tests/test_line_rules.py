"""Lines per block of the whole-line kernels (mfix_amd/csrc/leq_line.h), on the
host: what a block asks for leaves room for the blocks that the rules count on,
and the entries of streamed lines hold every line once."""
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]

PROGRAM = r"""
#include <cstdio>
#include "leq_line.h"
using namespace mfix;
int main() {
    const int64_t counts[] = {1, 2, 33, 255, 256, 513, 1025, 2178, 3528, 7169, 7320, 11325, 20000, 33282, 100000};
    for (size_t elem : {sizeof(double), sizeof(float)})
        for (int n = 3; n <= kWholeRows; ++n)
            for (int64_t lines : counts)
                for (int pin : {0, 16, 64}) {
                    const int lpb = whole_lpb(n, lines / whole_at_once(n, elem), elem, pin);
                    const size_t bytes = whole_elems(n, lpb) * elem + kWholeFixed;
                    if (lpb < 1 || lpb > kWholeLines || lpb * n > kWholeRows || bytes > 64 * 1024 ||
                        (!pin && lpb > 1 && 4 * bytes > 160 * 1024))
                        std::printf("whole %zu n %d lines %lld pin %d: %d lines, %zu bytes\n", elem, n, (long long)lines,
                                    pin, lpb, bytes);
                    if (!pin && elem == 8 && !line_streams(n, lines, 1000) && lines <= 65536 &&
                        (lines + lpb - 1) / lpb > kNumCus * kWholePerCu)
                        std::printf("rounds: n %d lines %lld: %d a block\n", n, (long long)lines, lpb);
                }
    for (int n = 3; n <= kWholeRows; ++n)
        for (int64_t lines : counts) {
            const int64_t ent = stream_entries(n, lines);
            const uint64_t step = entry_step(lines, ent);
            const int lpb = (int)((step + 0xffffffffull) >> 32);
            int64_t at = 0;
            bool ok = lpb <= kWholeLines && lpb * n <= kStreamRows &&
                      (size_t)stream_elems(n, lpb) * 8 <= kStreamLdsTarget && ent % kStreamBlocks == 0;
            for (int64_t j = 0; j < ent; ++j) {
                const int64_t a = entry_first(step, (int)j), b = entry_first(step, (int)j + 1);
                ok = ok && a == at && b >= a && b - a <= lpb;
                at = b;
            }
            if (!ok || at < lines) std::printf("stream: n %d lines %lld: %d an entry\n", n, (long long)lines, lpb);
        }
    return 0;
}
"""


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    from mfix_amd.build import HIP_FLAGS, _hipcc
    d = tmp_path_factory.mktemp("rules")
    (d / "rules.hip").write_text(PROGRAM)
    flags = [f for f in HIP_FLAGS if f not in ("-O3", "-fopenmp")]
    subprocess.run([_hipcc(), *flags, "-O1", "--offload-host-only", f"-I{ROOT / 'mfix_amd' / 'csrc'}", "-c",
                    str(d / "rules.hip"), "-o", str(d / "rules.o")], check=True)
    subprocess.run([_hipcc(), str(d / "rules.o"), "-o", str(d / "rules")], check=True)
    return d / "rules"


def test_blocks_fit(program):
    out = subprocess.run([str(program)], capture_output=True, text=True, timeout=100)
    assert out.returncode == 0 and out.stdout == ""
