"""The build's check of the hand-written loads into LDS: five wait states between a vector
instruction's write of a scalar register (a spilled one's way back) and the load's use of it, along
every path.  The compiler's hazard pass does not look into inline assembly."""
import importlib.util
import os

import pytest

PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "ring-sliding-window-attention_amd")
spec = importlib.util.spec_from_file_location("rswa_build", os.path.join(PKG, "build.py"))
build = importlib.util.module_from_spec(spec)
spec.loader.exec_module(build)

LOAD = ["s_nop 0", "buffer_load_dwordx4 v4, s[0:3], s9 offen lds"]


def _gap(n):
    return ["s_add_i32 s50, s50, 1"] * n


@pytest.mark.parametrize("write", ["v_readlane_b32 s2, v210, 7", "v_readfirstlane_b32 s9, v1",
                                   "v_readlane_b32 m0, v210, 7", "v_cmp_lt_i32_e64 s[0:1], v1, v2",
                                   "v_add_co_u32_e64 v1, s[2:3], v1, v2"])
def test_a_write_closer_than_five_states_is_found(write):
    assert build.close_sgpr_writes([write, *_gap(3), *LOAD])
    assert not build.close_sgpr_writes([write, *_gap(4), *LOAD])
    assert not build.close_sgpr_writes([write, "s_nop 3", *LOAD])
    # around a branch, and over the end of a loop
    assert build.close_sgpr_writes([write, "s_cbranch_scc1 L0", *_gap(9), "<L0>:", *_gap(2), *LOAD])
    assert not build.close_sgpr_writes([write, "s_cbranch_scc1 L0", *_gap(9), "<L0>:", *_gap(3), *LOAD])
    assert build.close_sgpr_writes(["<L1>:", *LOAD, write, "s_cbranch_vccnz L1"])
    assert not build.close_sgpr_writes([write, "s_branch L2", *LOAD])


def test_other_registers_are_let_be():
    for other in ("v_readlane_b32 s4, v210, 7", "v_readlane_b32 s10, v210, 7", "v_mul_f32_e32 v4, s2, v4",
                  "s_mov_b32 s2, s20", "v_add_co_u32_e64 v1, s[4:5], v1, v2"):
        assert not build.close_sgpr_writes([other, *LOAD])


def test_a_load_right_behind_a_write_of_m0_is_found():
    load = "buffer_load_dwordx4 v4, s[0:3], s9 offen offset:1024 lds"
    assert build.close_m0_writes(["s_mov_b32 m0, s5", load])
    assert build.close_m0_writes(["s_add_i32 m0, s5, 64", "<L0>:", load])
    assert not build.close_m0_writes(["s_mov_b32 m0, s5", "s_nop 0", load])
    assert not build.close_m0_writes(["s_mov_b32 m0, s5", "v_add_u32_e32 v1, v2, v3", load])
    assert not build.close_m0_writes(["s_mov_b32 s50, m0", load])
