"""How attention launches of few segments deal their blocks to the eight XCDs (``attn_deal.h``, compiled for the host): every block
once, in contiguous ranges, and no XCD with more than one block above another, whatever the heads and lengths."""

import shutil
import subprocess

import pytest

from come_amd.build import CSRC

DRIVER = r"""
#include <cstdio>
#include <cstdlib>
#include "attn_deal.h"
// argv: items of the lists in the order in which they are dealt; prints the blocks of every XCD, -1 for a range that is wrong
int main(int argc, char **argv) {
    int load[8] = {}, dealt = 0, all = 0;
    for (int i = 1; i < argc; ++i) {
        const int items = std::atoi(argv[i]);
        int next = 0;
        for (int x = 0; x < 8; ++x) {
            const come::XcdShare s = come::share_of(items, dealt, x);
            if (s.first != next || come::items_to(all, 0, dealt, x) != load[x]) load[x] = -1000000000;
            next = s.first + s.count;
            load[x] += s.count;
        }
        if (next != items) load[0] = -1000000000;
        dealt += items & 7;
        all += items;
    }
    for (int x = 0; x < 8; ++x) std::printf("%d ", load[x]);
}
"""


@pytest.fixture(scope="module")
def loads(tmp_path_factory):
    compiler = shutil.which("g++") or shutil.which("clang++")
    if compiler is None:
        pytest.skip("no host compiler")
    folder = tmp_path_factory.mktemp("deal")
    (folder / "deal.cpp").write_text(DRIVER)
    subprocess.run([compiler, "-std=c++17", f"-I{CSRC}", str(folder / "deal.cpp"), "-o", str(folder / "deal")], check=True)
    return lambda lists: [int(n) for n in subprocess.run([str(folder / "deal"), *map(str, lists)], check=True, capture_output=True, text=True).stdout.split()]


def lists_of(heads, lengths, block=128):
    """Blocks of all heads: the full ones of every segment, the longest first, then the last ones of at most 128 queries."""
    lengths = sorted(lengths, reverse=True)
    short = [0 < n % block <= 128 for n in lengths]
    return [heads * (-(-n // block) - s) for n, s in zip(lengths, short)] + [heads * s for s in short]


@pytest.mark.parametrize("block", [128, 256, 512])
@pytest.mark.parametrize("heads", [1, 3, 4, 5, 6, 7, 8, 12, 16])
def test_no_xcd_has_more_than_one_block_above_another(loads, heads, block):
    for lengths in ([801] * 3, [954] * 5, [435] * 5, [3344] * 3, [200] * 8, [1], [7000, 5000], [453, 355, 411, 430, 443], [900, 0, 1, 129, 128]):
        lists = lists_of(heads, lengths, block)
        got = loads(lists)
        assert sum(got) == sum(lists) and max(got) - min(got) <= 1, (lengths, got)


def test_one_round_stays_one_round(loads):
    # launches whose 128-query workgroups have a CU each, 32 an XCD
    for heads, lengths in ((12, [801] * 3), (6, [954] * 5), (12, [435] * 5), (6, [782] * 6)):
        assert max(loads(lists_of(heads, lengths))) <= 32
