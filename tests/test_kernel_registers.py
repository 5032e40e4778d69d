"""Registers of kernels whose launches count on all of their workgroups being resident, as the built library's code objects state them."""
import os
import re
import subprocess

import pytest

from test_dpp_wait_states import TOOLS, built_library, code_objects


@pytest.mark.parametrize("kernel", ["adam_kernelILb1E", "adam_pair_kernelILb1E"])
def test_all_workgroups_of_an_optimisers_launch_are_resident(tmp_path, kernel):
    """A launch has up to 960 workgroups (csrc/optim.hip), four for each of 256 compute units; of five wavefronts each that is five to a SIMD, whose 512 registers a lane are given out in eights.
    With the registers for blocks of sums, which these instances never add up, it was three workgroups to a compute unit and a second round: 2,000,000 elements 13.1 us instead of 9.5."""
    used = []
    for code in code_objects(built_library(), tmp_path):
        notes = subprocess.run([os.path.join(TOOLS, "llvm-readelf"), "--notes", code], check=True, capture_output=True, text=True).stdout
        name = ""
        for field in re.findall(r"\.(name|vgpr_count):\s+(\S+)", notes):      # in this order for each kernel
            if field[0] == "name":
                name = field[1]
            elif kernel in name:
                used.append(int(field[1]))
    assert len(used) == 1 and -(-used[0] // 8) * 8 * 5 <= 512, used
