"""Entry points that may allocate device memory, create events or capture a graph select their
context's device first: the caller's current device may be another one (read from the source;
a second device is not needed to see it)."""
import os
import re

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "cardiomechanics_amd", "csrc")
# what allocates: directly, or below these internal functions (first solves set up their workspace)
ALLOCATES = re.compile(r"\b(alloc|upload|newton|krylov|bnewton|eval_elements|build_damping|tune_spmv)\s*\(|DevBuf|hipEvent")


@pytest.mark.parametrize("source", ["cmg_api.hip", "batch.hip", "mlp.hip", "noalloc.hip"])
def test_allocating_entry_points_select_their_device(source):
    with open(os.path.join(CSRC, source)) as f:
        functions = re.findall(r"^int (cmg_\w+)\([^)]*\) \{\n(.*?)^\}\n", f.read(), re.S | re.M)
    assert functions
    late = []
    for name, body in functions:
        first = ALLOCATES.search(body)
        select = body.find("hipSetDevice(")
        if first and not 0 <= select < first.start():
            late.append(name)
    assert late == []
