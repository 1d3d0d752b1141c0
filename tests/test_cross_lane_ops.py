"""Cross-lane operations read other lanes' registers, whose value is undefined
where those lanes are masked off: none may stand behind a short-circuit
operator, which masks them off lane by lane."""
import glob
import os
import re

import pytest

CSRC = os.path.join(os.path.dirname(os.path.abspath(__file__)), "..", "openlowdin_amd", "csrc")
FILES = [f for ext in ("h", "hip", "cpp") for f in sorted(glob.glob(os.path.join(CSRC, "*." + ext)))]
BEHIND = re.compile(r"(\|\||&&|\?)[^;{}]*?\b(__shfl\w*|__ballot|wave_sum|group_sum|row_sum|wave_total|"
                    r"__builtin_amdgcn_(update_dpp|mov_dpp|ds_bpermute|ds_swizzle))\s*[<(]", re.S)


@pytest.mark.parametrize("path", FILES, ids=[os.path.basename(f) for f in FILES])
def test_no_cross_lane_operation_behind_a_short_circuit(path):
    text = open(path).read()
    text = re.sub(r"//[^\n]*|/\*.*?\*/", " ", text, flags=re.S)
    hits = [m.group(0) for statement in text.split(";") for m in BEHIND.finditer(statement)]
    assert not hits, hits
