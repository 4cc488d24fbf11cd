"""Every kernel that stages a table in LDS has a workgroup barrier before it looks
anything up there.  The stage is written by all threads of the workgroup, so
without the barrier a fast wave reads entries that a slow one has not written:
wrong integrals now and then, which a run on a GPU hardly ever shows.  Checked in
the sources."""
import glob
import os
import re

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "rchem_amd", "csrc")


def _stages(text):
    """(table, code from the stage to the table's first use as an argument)."""
    text = re.sub(r"//[^\n]*", "", text)
    for m in re.finditer(r"\bstage_boys<[^;]*?>\((\w+),[^;]*;", text):
        table = m.group(1)
        rest = text[m.end():]
        use = re.search(r"\w[\w<>:, ]*\([^;]*?,\s*" + table + r"\s*[,)]", rest)
        assert use, f"{table} is staged and never passed on"
        # up to the use itself, not to the start of the call it is found in
        yield table, rest[:use.end()]


@pytest.mark.parametrize("path", sorted(p for p in glob.glob(os.path.join(CSRC, "*.h*"))
                                        if os.path.basename(p) != "boys.hpp"
                                        and "stage_boys<" in open(p).read()), ids=os.path.basename)
def test_barrier_between_stage_and_first_lookup(path):
    for table, code in _stages(open(path).read()):
        assert "__syncthreads()" in code, f"{os.path.basename(path)}: {table} read before a barrier"


def test_the_check_sees_a_missing_barrier():
    bad = "stage_boys<L>(tab, a.t);\n for (;;) run<L>(x, tab, y);\n __syncthreads();"
    (table, code), = _stages(bad)
    assert table == "tab" and "__syncthreads()" not in code
