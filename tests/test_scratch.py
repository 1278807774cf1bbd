"""What the compiler spills in the dQ kernel of head dim 64, the form closest to the end of its registers: a reload inside the loop waits
for the tile copies in flight, so that a launch gets slower without any result to tell it by."""

import os
import re
import shutil
import subprocess

import pytest

from cornstarch_amd import build
from tests.test_copy_hazard import LLVM, _code_objects

# mangled: type, head dim 64, mask mode, bias form (0 none, 1 read group by group, 2 with the tiles), several passes, streams
DQ = re.compile(r"13bwd_dq_kernelI\w*?Li64ELi([012])ELi([012])ELb([01])ELi[12]EE")


def spilled(notes):
    """(mask mode, bias form, several passes, spilled vector registers) of every dQ instantiation of head dim 64."""
    found = []
    for kernel in re.split(r"\n\s*- \.agpr_count", notes)[1:]:
        form = DQ.search(re.search(r"\.name:\s+(\S+)", kernel)[1])
        if form:
            found.append((*map(int, form.groups()), int(re.search(r"\.vgpr_spill_count:\s+(\d+)", kernel)[1])))
    return found


def test_dq_spills_no_more_than_it_has_to(tmp_path):
    if shutil.which("llvm-readelf", path=LLVM) is None or not os.path.exists(build.LIB_PATH):
        pytest.skip("needs the built library and the LLVM tools it is built with")
    found = []
    for i, code in enumerate(_code_objects(build.LIB_PATH, str(tmp_path))):
        path = tmp_path / f"{i}.co"
        path.write_bytes(code)
        found += spilled(subprocess.run([f"{LLVM}/llvm-readelf", "--notes", str(path)], capture_output=True, text=True, check=True).stdout)
    assert len(found) == 2 * 3 * 3 * 3  # types, mask modes, bias forms; one stream, two, several passes
    # several passes over 64-bit row addresses: 33 as compiled, 101 over masks (which gain more by what takes them), 48 with a bias
    # that is read group by group
    for mode, bias, passes, count in found:
        assert count <= (0 if not passes or bias == 2 else 48 if bias else 104 if mode == 2 else 36), (mode, bias, passes)
