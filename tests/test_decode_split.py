"""The rule for a decode launch's automatic work split (csrc/kvc_decode_split.h),
on the CPU.  Expected chunk lengths (in 32-token blocks) are the measured ones:
never slower than chunks of 4 blocks, which every launch of up to 1024 blocks
took before the rule."""
import shutil
import subprocess
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parents[1] / "qwen3.5-9b-bfp8b-1xn300_amd" / "csrc"
CXX = shutil.which("g++")
pytestmark = pytest.mark.skipif(CXX is None, reason="needs g++")

# stdin: one launch a line, the sequences' block counts; stdout: blocks per chunk
PROGRAM = r"""
#include <cstdio>
#include <iostream>
#include <sstream>
#include <string>
#include <vector>
#include "kvc_decode_split.h"
int main() {
    std::string line;
    while (std::getline(std::cin, line)) {
        std::istringstream in(line);
        std::vector<int32_t> nb;
        for (int x; in >> x;) nb.push_back(x);
        std::printf("%d\n", kvc::auto_chunk_blocks(nb.data(), (int32_t)nb.size(), false));
    }
}
"""


@pytest.fixture(scope="module")
def picks(tmp_path_factory):
    d = tmp_path_factory.mktemp("decode_split")
    (d / "split.cpp").write_text(PROGRAM)
    subprocess.run([CXX, "-O2", "-std=c++17", "-Wall", "-Wextra", f"-I{CSRC}", str(d / "split.cpp"), "-o",
                    str(d / "split")], check=True)

    def run(launches):
        text = "\n".join(" ".join(map(str, nb)) for nb in launches)
        out = subprocess.run([str(d / "split")], input=text, capture_output=True, text=True, check=True).stdout
        return [int(line) for line in out.split()]

    return run


MEASURED = [
    # block counts, blocks per chunk
    ([3, 1, 2], 3), ([4], 1), ([10], 1), ([32], 1), ([128], 4),
    ([4] * 6, 1),                              # exchanging pays for a few sequences
    ([4] * 10, 4), ([4] * 13, 4), ([4] * 32, 4), ([4, 1, 2, 3] * 12, 4),  # one chunk per sequence
    ([18] * 4, 2), ([29] * 3, 2), ([32] * 3, 2), ([16] * 8, 2),
    ([35] * 2, 3), ([43] * 2, 3), ([50] * 2, 4), ([64] * 2, 4), ([38] * 3, 4), ([45, 40, 6], 3),
    ([43] * 3, 3), ([63] * 3, 3), ([10] * 64, 10), ([32] * 64, 32),
]


@pytest.mark.parametrize("blocks,cb", MEASURED)
def test_chunk_length(picks, blocks, cb):
    assert picks([blocks]) == [cb]


def test_chunk_counts(picks):
    """At most 32 chunks per sequence; one round of at most 64 chunks unless
    that leaves one chunk too long for the rest to fill."""
    launches = [[a] * n + [b] * m for a in (1, 4, 5, 40, 300) for b in (1, 7, 64, 1000) for n in (0, 1, 5, 40)
                for m in (1, 3, 24)]
    for nb, cb in zip(launches, picks(launches)):
        chunks = sum(-(-x // cb) for x in nb)
        short = max(4, round(0.25 * sum(nb) ** 0.5))
        assert 1 <= cb and (chunks <= 64 or cb == short), nb
        assert max(-(-x // cb) for x in nb) <= 32 or cb == short, nb
