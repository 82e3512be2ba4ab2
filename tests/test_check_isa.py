"""The build's check of the device assembly (gcnasm_amd/csrc/check_isa.py) on small made-up kernels: a vector instruction that
writes an MFMA's operand in the two slots in front of it is found on every path, a loop's back edge among them."""
import os
import sys

import pytest

sys.path.insert(0, os.path.join(os.path.dirname(os.path.abspath(__file__)), "..", "gcnasm_amd", "csrc"))
import check_isa

MFMA = "v_mfma_f32_16x16x128_f8f6f4 a[0:3], v[8:15], v[16:23], a[0:3]"


def _check(tmp_path, *body):
    text = "\n".join(["_Z1xgemm_a8w8_widev:", *body, "v_accvgpr_read_b32 v0, a[0]", "buffer_store_dwordx4 v[0:3], v4, s[0:3], 0 offen", "s_nop 1", "s_endpgm", ""])
    path = tmp_path / "x.s"
    path.write_text("\t.text\n" + text)
    check_isa.main(str(path))


@pytest.mark.parametrize("gap", [0, 1, 2])
def test_straight_line(tmp_path, gap):
    body = ["v_mov_b32_e32 v9, 0", *["s_nop 0"] * gap, MFMA]
    if gap < 2:
        with pytest.raises(SystemExit, match="directly in front"):
            _check(tmp_path, *body)
    else:
        _check(tmp_path, *body)


@pytest.mark.parametrize("writes", ["v_mov_b32_e32 v17, v2", "v_mov_b32_e32 v7, v2"])
def test_back_edge(tmp_path, writes):
    """The instruction in front of the branch back is one slot further off than the branch."""
    body = ["s_nop 0", "s_nop 0", ".LBB0_1:", MFMA, "s_waitcnt vmcnt(0)", "s_barrier", writes, "s_cbranch_scc1 .LBB0_1", "s_nop 7"]
    if "v17" in writes:
        with pytest.raises(SystemExit, match="directly in front"):
            _check(tmp_path, *body)
    else:
        _check(tmp_path, *body)


def test_nothing_falls_through_an_unconditional_branch(tmp_path):
    _check(tmp_path, "s_branch .LBB0_2", "v_mov_b32_e32 v9, 0", "s_branch .LBB0_3", ".LBB0_2:", MFMA, ".LBB0_3:", "s_nop 7")
