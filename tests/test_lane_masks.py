"""No unit has a vector copy or spill ahead of the instruction that widens the lane mask where lanes join again (the lanes that
join would lose the value)."""
import importlib.util
import os

import pytest

SPEC = importlib.util.spec_from_file_location("mrl_build", os.path.join(os.path.dirname(__file__), "..", "mojo-rl_amd", "build.py"))
build = importlib.util.module_from_spec(SPEC)
SPEC.loader.exec_module(build)

JOIN = """name:            kernel
  bb.1:
    liveins: $vgpr0
    %s
    $exec = S_OR_B64 $exec, killed renamable $sgpr2_sgpr3, implicit-def $scc
    renamable $vgpr4 = COPY $vgpr0, implicit $exec
  bb.2:
    renamable $vgpr5 = COPY $vgpr0, implicit $exec
    $exec = S_AND_B64 $exec, $sgpr4_sgpr5, implicit-def $scc
"""


@pytest.mark.parametrize("ahead,fault", [
    ("renamable $vgpr7 = COPY $vgpr6, implicit $exec", True),
    ("$vgpr7 = V_MOV_B32_e32 $vgpr6, implicit $exec", True),
    ("SI_SPILL_V32_SAVE killed $vgpr7, %stack.3, $sgpr32, 0, implicit $exec", True),
    ("$agpr3 = V_ACCVGPR_WRITE_B32_e64 $vgpr6, implicit $exec", True),
    ("$vgpr255 = SI_SPILL_S32_TO_VGPR killed $sgpr13, 1, killed $vgpr255", False),
    ("$sgpr2 = SI_RESTORE_S32_FROM_VGPR $vgpr255, 1", False),
    ("$vgpr255 = IMPLICIT_DEF", False),
    ("renamable $sgpr2_sgpr3 = COPY $sgpr6_sgpr7", False),
])
def test_what_the_search_finds(ahead, fault):
    joins, faults = build.narrow_copies((JOIN % ahead).splitlines())
    assert joins == 1 and len(faults) == int(fault)


def test_no_vector_copy_ahead_of_a_widening_mask():
    found = build.check_lane_masks()
    for unit, (joins, faults) in found.items():
        print(unit, joins, flush=True)
        assert not faults, (unit, faults[:5])
    assert sum(joins for joins, _ in found.values()) > 10000   # (the dumps were what the search reads)
