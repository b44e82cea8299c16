"""The rule for a prefill launch's work split (csrc/kvc_prefill_split.h), on the
CPU: one workgroup runs per CU, so whole rounds of workgroups count.

Expected picks are the measured ones (us per layer, kvc_prefill_attn and
kvc_prefill_step with 32- and with 16-row workgroups; 13 sequences of 100 rows
with nothing cached 17.0 against 21.9 and 24.2 against 29.7)."""
import shutil
import subprocess
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parents[1] / "qwen3.5-9b-bfp8b-1xn300_amd" / "csrc"
CXX = shutil.which("g++")
pytestmark = pytest.mark.skipif(CXX is None, reason="needs g++")

# stdin: one launch a line, "n_q prefix prefix ..."; stdout: rows, tiles per
# piece, and the partials that the pieces take against their limit
PROGRAM = r"""
#include <cstdio>
#include <iostream>
#include <sstream>
#include <string>
#include "kvc_prefill_split.h"
int main() {
    std::string line;
    while (std::getline(std::cin, line)) {
        std::istringstream in(line);
        kvc::PrefillArgs a{};
        in >> a.n_q;
        for (int p; in >> p;) a.q_pos0[a.n_seqs++] = p;
        a.n_groups = a.n_seqs * kvc::kKvHeads;
        kvc::prefill_split(a);
        long slots = 0;
        const long blocks = (a.n_q + a.rows - 1) / a.rows;
        for (int j = 0; a.piece_tiles && j < a.n_seqs; j++) {
            const long tiles = (a.q_pos0[j] + a.n_q + kvc::kPfKeys - 1) / kvc::kPfKeys;
            slots += (tiles + a.piece_tiles - 1) / a.piece_tiles * kvc::kKvHeads * blocks;
        }
        std::printf("%d %d %ld %ld\n", a.rows, a.piece_tiles, slots, (long)kvc::pf_max_parts(a.rows));
    }
}
"""


@pytest.fixture(scope="module")
def picks(tmp_path_factory):
    d = tmp_path_factory.mktemp("prefill_split")
    (d / "split.cpp").write_text(PROGRAM)
    subprocess.run([CXX, "-O2", "-std=c++17", "-Wall", "-Wextra", f"-I{CSRC}", str(d / "split.cpp"), "-o",
                    str(d / "split")], check=True)

    def run(launches):
        text = "\n".join(" ".join(map(str, (n_q, *prefix))) for n_q, prefix in launches)
        out = subprocess.run([str(d / "split")], input=text, capture_output=True, text=True, check=True).stdout
        return [tuple(map(int, line.split())) for line in out.splitlines()]

    return run


MEASURED = [
    # n, n_q, prefix of each sequence, rows per workgroup that was faster, unsplit
    (10, 100, 0, 32), (13, 100, 0, 32), (16, 80, 0, 32), (12, 112, 0, 32), (18, 64, 0, 32), (24, 48, 0, 32),
    (33, 32, 0, 32), (9, 128, 0, 32), (7, 200, 0, 32), (32, 48, 0, 32), (13, 100, 80, 32), (18, 64, 80, 32),
    (24, 48, 80, 32), (9, 128, 80, 32), (50, 20, 0, 32), (64, 32, 0, 32), (8, 250, 0, 32),
    (1, 500, 0, 16), (6, 30, 0, 16), (16, 20, 0, 16), (2, 64, 0, 16), (64, 16, 80, 16), (40, 33, 0, 16),
]


@pytest.mark.parametrize("n,n_q,prefix,rows", MEASURED)
def test_unsplit_rows(picks, n, n_q, prefix, rows):
    assert picks([(n_q, [prefix] * n)])[0][:2] == (rows, 0)


def test_equal_workgroups_count_whole_rounds(picks):
    """Sequences of one key tile: 16-row workgroups are never taken for more
    rounds than 32-row ones need."""
    launches = [(n_q, [0] * n) for n in range(1, 65) for n_q in range(1, 65)]
    for (n_q, prefix), (rows, piece, _, _) in zip(launches, picks(launches)):
        rounds = {r: -(-4 * len(prefix) * -(-n_q // r) // 256) for r in (16, 32)}
        assert piece == 0
        assert rows == 32 or rounds[16] <= rounds[32], (len(prefix), n_q)


def test_long_keys_are_cut_within_the_workspace(picks):
    launches = [(32, [4001]), (128, [16000]), (128, [1000]), (16, [100 * i for i in range(1, 41)]), (1, [32000] * 20),
                (3, [100000] * 3)]
    for (n_q, prefix), (rows, piece, slots, most) in zip(launches, picks(launches)):
        assert piece > 0 and slots <= most, (n_q, prefix)


def test_routes_of_the_gpu_cases(picks):
    from test_gpu_prefill_split import CASES

    for case, (rows, piece, _, _) in zip(CASES, picks([(n_q, prefix) for prefix, n_q, _ in CASES])):
        assert (rows, piece > 0) == case[2], case
