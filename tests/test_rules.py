"""The host rules that choose a call's bf16 linears and the tiles' heights, compiled
for the CPU: the lines measured on an MI355X, that every call has exactly one
kernel, and that the heights follow the number of CUs."""
import shutil
import subprocess
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parent.parent / "hybridagent_amd" / "csrc"

PROGRAM = """
#include <cstdio>
#include "rules.hpp"
using namespace w4a16;
int main() {
  char what[16];
  long long a, b, c, d;
  while (scanf("%15s %lld %lld %lld %lld", what, &a, &b, &c, &d) == 5) {
    if (what[0] == 'f') printf("%d\\n", (int)ffn_fragment_rows(a, b, c, d & 1, d & 2));
    else if (what[0] == 'r') printf("%d\\n", (int)linear_tiled_rows(a, b, c));
    else if (what[0] == 'g') printf("%d\\n", gemm_bf16_blocks(a, b, c));
    else if (what[0] == 'l') printf("%d\\n", linear_w4_blocks(a, b, c, d));
    else return 1;
  }
}
"""


@pytest.fixture(scope="module")
def ask(tmp_path_factory):
    cxx = shutil.which("g++") or shutil.which("c++")
    if cxx is None:
        pytest.skip("no host compiler")
    d = tmp_path_factory.mktemp("rules")
    (d / "rules.cpp").write_text(PROGRAM)
    subprocess.run([cxx, "-std=c++17", "-O1", f"-I{CSRC}", str(d / "rules.cpp"), "-o", str(d / "rules")], check=True)

    def run(lines):
        out = subprocess.run([str(d / "rules")], input="\n".join(" ".join(map(str, x)) for x in lines), text=True,
                             capture_output=True, check=True)
        return [int(v) for v in out.stdout.split()]

    return run


# the kernel that was faster by more than 2 %, at H = 2816: streamed from fragment-order rows (1) or tiled (0)
MEASURED = [(65, 1056, 1), (65, 2112, 1), (65, 4096, 1), (128, 512, 1), (128, 2112, 1), (128, 4096, 1), (128, 6144, 1),
            (144, 1056, 1), (192, 512, 1), (192, 1056, 1), (256, 512, 1), (129, 4096, 0), (129, 6144, 0),
            (192, 4096, 0), (208, 1600, 0), (208, 2112, 0), (208, 3072, 0), (288, 1600, 0), (288, 2112, 0),
            (320, 1056, 0), (384, 512, 0), (2048, 2112, 0)]


def test_fragment_rows_where_they_are_faster(ask):
    got = ask([("f", M, 2816, Im, 3) for M, Im, _ in MEASURED])
    assert got == [want for _, _, want in MEASURED]


def test_fragment_rows_need_room_and_more_than_one_row_tile(ask):
    assert ask([("f", 16, 2816, 2112, 3), ("f", 17, 2816, 2112, 3), ("f", 64, 2816, 2112, 2),
                ("f", 2048, 2816, 2112, 1)]) == [0, 1, 0, 1]


def test_no_call_of_many_rows_streams_row_major(ask):
    # rows that fit are streamed in fragment order or tiled, never streamed row-major, from 17 rows on
    sizes = [(M, K, N) for M in (17, 64, 65, 128, 129, 200, 257, 500, 769, 2000, 9000) for K in (160, 1024, 2816)
             for N in (32, 160, 512, 2112)]
    frag = ask([("f", M, K, N, 3) for M, K, N in sizes])
    tiled = ask([("r", M, N, K, 0) for M, K, N in sizes])
    assert all(f or t for f, t in zip(frag, tiled))


def test_tile_heights_at_256_cus(ask):
    # the FFN block's gate/up (4224 weight rows) and down, Linear4Bit at 2816 x 2816
    assert ask([("g", 512, 4224, 256, 0), ("g", 1024, 4224, 256, 0), ("g", 2048, 4224, 256, 0),
                ("g", 2048, 2816, 256, 0), ("l", 2048, 2816, 256, 6), ("l", 4096, 2816, 256, 6),
                ("l", 4096, 2816, 256, 4)]) == [2, 3, 5, 3, 3, 6, 3]


@pytest.mark.parametrize("cus", [32, 64, 128, 256, 304])
def test_tile_heights_are_the_cheapest_for_the_cus(ask, cus):
    gemm, w4 = [2, 3, 4, 5, 6], [31, 37, 44, 52, 61, 72]
    sizes = [(M, n) for M in (65, 300, 1024, 2048, 4096) for n in (704, 2816, 4224)]
    got = ask([("g", M, n, cus, 0) for M, n in sizes] + [("l", M, n, cus, 6) for M, n in sizes])
    for (M, n), cost, mb in zip(sizes * 2, [gemm] * len(sizes) + [w4] * len(sizes), got):
        time = [-(-(-(-M // (32 * b)) * -(-n // 256)) // cus) * c for b, c in enumerate(cost, 1)]
        assert time[mb - 1] == min(time), (M, n, mb, time)
