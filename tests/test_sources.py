"""Rules the kernels' sources keep that no test of results shows."""
from __future__ import annotations

import glob
import os
import re

import pytest

from jacq_amd import build

CSRC = os.path.join(os.path.dirname(build.__file__), "csrc")
SOURCES = sorted(glob.glob(os.path.join(CSRC, "*.hip")) + glob.glob(os.path.join(CSRC, "*.h")))


def asm_statements(text):
    """The argument lists of the asm statements."""
    for m in re.finditer(r"\basm\b(?:\s+volatile)?\s*\(", text):
        depth, i = 1, m.end()
        while depth:
            depth += {"(": 1, ")": -1}.get(text[i], 0)
            i += 1
        yield text[m.end():i - 1]


def unwaited_loads(text):
    """asm statements that load into registers and do not wait for it themselves: the
    compiler takes the outputs as written, and may reuse them while the load is in
    flight."""
    load = re.compile(r"\b(global_load|buffer_load|flat_load|scratch_load|s_load|ds_read)(?!_lds)\w*")
    return [s for s in asm_statements(text)
            if load.search(s) and not re.search(r"s_waitcnt", s[load.search(s).end():])]


@pytest.mark.parametrize("path", SOURCES, ids=os.path.basename)
def test_asm_loads_wait_in_their_own_statement(path):
    assert not unwaited_loads(open(path).read())


def test_the_rule_finds_a_load_in_flight():
    late = 'asm volatile("global_load_dwordx4 %0, %1, off sc1" : "=v"(v) : "v"(p) : "memory");'
    assert unwaited_loads(late)
    assert not unwaited_loads(late.replace("sc1", "sc1\\n\\ts_waitcnt vmcnt(0)"))
    assert not unwaited_loads('asm("global_load_lds_dwordx4 %0, off" :: "v"(p));')


def test_the_build_refuses_spills_of_every_kernel_but_the_cross_check():
    """The VALU decode (kivi_decode.hip) is a cross-check whose speed is not followed."""
    kernels = set()
    for path in SOURCES:
        if os.path.basename(path) != "kivi_decode.hip":
            kernels |= set(re.findall(r"__global__[^;{]*?void\s+(?:__attribute__\S+\s+)?(\w+)\s*\(",
                                      open(path).read()))
    assert len(kernels) >= 3 and kernels == set(build.NO_SCRATCH)
