"""The entry points that one source file calls in others: declared once, where both sides include it, and as the loader knows them."""

from __future__ import annotations

import re
from ctypes import c_float, c_int, c_size_t, c_void_p

from tokasaurus_amd.kernels import build, library

HEADER = (build.CSRC / "calls.h").read_text()
DECLARED = {name: args for name, args in re.findall(r"TK_API int (\w+)\(([^;]*)\);", HEADER)}


def test_no_entry_point_is_declared_by_hand_where_it_is_called():
    calls = (build.CSRC / "block_calls.hip").read_text()
    assert 'extern "C"' not in calls and '#include "calls.h"' in calls
    assert set(re.findall(r"\btk_\w+(?=\()", calls)) - {"tk_block_calls"} <= set(DECLARED)
    for source in build.CSRC.glob("*.hip"):
        text = source.read_text()
        if any(re.search(rf"TK_API int {name}\(", text) for name in DECLARED):
            assert '#include "calls.h"' in text, source.name


def test_the_loader_knows_them_with_these_arguments():
    kinds = {"int": c_int, "float": c_float, "size_t": c_size_t}
    for name, args in DECLARED.items():
        types = [c_void_p if "*" in a or "hipStream_t" in a else kinds[a.split()[0]] for a in args.split(",")]
        assert types == library._SIGNATURES[library._GROUP_OF[name]][name], name
