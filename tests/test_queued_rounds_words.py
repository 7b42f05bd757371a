"""The queued rounds' launches (mid.hip) share one small state.  A launch that
tests a word of it before its barriers must not store that word: a block that
starts late would have waves that read the old value and waves that read the
new one and leave, and the ones that stay would go on over shared memory the
others never wrote.  Read off the source: for every kernel with a barrier, the
outcome words of *st (those that make launches leave) that it loads and those
that it stores are different ones."""
import os
import re

import pytest

OUTCOMES = {"stop", "found", "ended", "skewed"}
SRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "rama_amd", "csrc", "mid.hip")


def _kernels():
    with open(SRC) as f:
        text = re.sub(r"//[^\n]*", "", f.read())
    return re.findall(r"__global__[^;{]*?\b(k_mid_\w+)\(MidArgs a[^)]*\)\s*\{(.*?)\n\}", text, re.S)


def _words(body):
    stores = set(re.findall(r"\bst->(\w+)\s*=(?!=)", body)) | set(re.findall(r"_(?:store|fetch_or)\(&st->(\w+)", body))
    rest = re.sub(r"\bst->\w+\s*=(?!=)", "", body)
    rest = re.sub(r"_(?:store|fetch_or)\(&st->\w+", "", rest)
    return set(re.findall(r"\bst->(\w+)", rest)), stores


def test_kernels_are_found():
    names = [n for n, _ in _kernels()]
    for k in ("begin", "cycles", "pick", "resolve", "keys", "scatter", "bucket", "finish"):
        assert "k_mid_" + k in names


@pytest.mark.parametrize("name,body", _kernels(), ids=lambda x: x if x.startswith("k_mid_") else "")
def test_no_launch_stores_a_word_it_tests(name, body):
    loads, stores = _words(body)
    if "__syncthreads" in body or "block_" in body or "combine_partials" in body:
        both = loads & stores & OUTCOMES
        assert not both, "%s loads and stores %s" % (name, sorted(both))
