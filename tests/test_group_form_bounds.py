"""The kernel that forms a group (bpt_amd/csrc/bptplan.hip, k_group_form) clears its array of member masks, two entries a word, while it
loads the records.  This replays the loop with the condition and the array's size taken from the kernel's source, for every number
of records a group may have: every word that an entry's mask can land in is cleared, and none outside the array.  CPU only."""
import os
import re

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SRC = open(os.path.join(ROOT, "bpt_amd", "csrc", "bptplan.hip")).read()
KERNEL = SRC[SRC.index("void k_group_form("):]
CAPS = sorted({int(x) for x in re.findall(r"k_group_form<(\d+),", SRC)})


def test_sizes_the_kernel_is_compiled_for():
    assert CAPS == [1024, 2048, 4096] and int(re.search(r"GRP_MAX_EDGES = (\d+);", SRC).group(1)) == CAPS[-1]


@pytest.mark.parametrize("cap", CAPS)
def test_cleared_words_are_those_of_the_entries(cap):
    words = eval(re.search(r"emask2\[(CAP / \d+)\];", KERNEL).group(1).replace("/", "//"), {"CAP": cap})
    cleared_if = compile(re.search(r"if \(([^()]+)\) emask2\[t\] = 0;", KERNEL).group(1), "cleared_if", "eval")
    for n in [*range(1, 140), *range(cap - 20, cap + 1)]:
        padded = max(128, 1 << (n - 1).bit_length())             # the loop's end: the keys that are sorted
        assert padded <= cap
        last = max(t for t in range(padded) if eval(cleared_if, {"t": t, "n": n}))
        assert all(eval(cleared_if, {"t": t, "n": n}) for t in range(last))
        assert last < words, f"{n} records clear word {last} of {words}"
        assert last >= (n - 1) >> 1, f"{n} records leave the word of the last entry uncleared"
