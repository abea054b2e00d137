"""The check that the build makes of its generated assembly (csrc/asm_lint.py) on small pieces of it: direct-to-LDS loads that some path
through a kernel never waits for, and the two hazards in front of a load."""

import pytest

from lorafusion_amd.csrc.asm_lint import lint

LOAD = "\tbuffer_load_dwordx4 v1, s[0:3], s9 offen lds\n"


def _found(tmp_path, body):
    path = tmp_path / "k.s"
    path.write_text("\t.text\nkernel:                ; @kernel\n" + body + "\ts_endpgm\n\t.section x\n.Lfunc_end0:\n\t.size kernel, 4\n")
    return lint(str(path))


@pytest.mark.parametrize("body,bad", [
    (LOAD, True),
    (LOAD + "\ts_waitcnt vmcnt(0)\n", False),
    (LOAD + "\ts_waitcnt vmcnt(0) lgkmcnt(0)\n", False),
    (LOAD + "\ts_waitcnt lgkmcnt(0)\n", True),
    (LOAD + "\tglobal_load_dword v2, v3, s[4:5]\n\ts_waitcnt vmcnt(1)\n", False),          # the load is the older of two
    (LOAD + "\tglobal_load_dword v2, v3, s[4:5]\n\ts_waitcnt vmcnt(2)\n", True),
    ("\tglobal_load_dword v2, v3, s[4:5]\n", False),                                         # not to LDS
    ("\ts_cbranch_scc1 .LBB0_2\n" + LOAD + "\ts_waitcnt vmcnt(0)\n.LBB0_2:\n", False),
    (LOAD + "\ts_cbranch_scc1 .LBB0_2\n\ts_waitcnt vmcnt(0)\n.LBB0_2:\n", True),              # waited for on one of two paths
    (LOAD + "\ts_cbranch_scc1 .LBB0_2\n\ts_waitcnt vmcnt(0)\n\ts_endpgm\n.LBB0_2:\n", True),   # ... that end on their own
    (".LBB0_1:\n" + LOAD + "\ts_cbranch_scc1 .LBB0_1\n\ts_waitcnt vmcnt(0)\n", False),
    (LOAD + "\ts_waitcnt vmcnt(0)\n\ts_branch .LBB0_3\n" + LOAD + ".LBB0_3:\n", False),         # the second load is never reached
])
def test_loads_left_open(tmp_path, body, bad):
    assert any("never waited for" in v for v in _found(tmp_path, body)) == bad


def test_hazards_in_front_of_a_load(tmp_path):
    wait = "\ts_waitcnt vmcnt(0)\n"
    assert any("needs 5" in v for v in _found(tmp_path, "\tv_readlane_b32 s9, v4, 1\n" + LOAD + wait))
    assert not _found(tmp_path, "\tv_readlane_b32 s9, v4, 1\n\ts_nop 4\n" + LOAD + wait)
    assert any("M0 needs" in v for v in _found(tmp_path, "\ts_mov_b32 m0, s7\n" + LOAD + wait))
    assert not _found(tmp_path, "\ts_mov_b32 m0, s7\n\ts_nop 0\n" + LOAD + wait)
