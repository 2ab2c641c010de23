"""The build's check of the code generated around hand-scheduled loads: it passes on what a
good build looks like and names each kind of break."""
import os

import pytest

from ferrum_amd import build, isa_check

GOOD = """
	.text
_Z6kernelv:
	s_load_dwordx2 s[0:1], s[4:5], 0x0
	;;#ASMSTART
	global_load_dwordx2 v[4:5], v[2:3], off
	;;#ASMEND
	v_add_u32_e32 v9, v8, v7
	;;#ASMSTART
	s_mov_b32 m0, s3
	s_nop 0
	global_load_lds_dwordx4 v[2:3], off
	;;#ASMEND
	s_add_u32 s2, s2, 1
	;;#ASMSTART
	s_waitcnt vmcnt(1)
	;;#ASMEND
	v_mov_b32_e32 v6, v4
	global_load_dword v10, v[2:3], off
	s_endpgm
.Lfunc_end0:
	.amdhsa_kernel _Z6kernelv
		.amdhsa_private_segment_fixed_size 0
	.end_amdhsa_kernel
"""


def test_a_clean_kernel_passes():
    assert isa_check.violations(GOOD) == []


@pytest.mark.parametrize("old,new,message", [
    # a copy of the destination before the wait
    ("v_add_u32_e32 v9, v8, v7", "v_mov_b32_e32 v9, v5", "touches registers loaded"),
    # a load of the compiler's own between the counted loads and the wait
    ("s_add_u32 s2, s2, 1", "global_load_dword v11, v[2:3], off", "hand-counted wait"),
    # the compiler keeps something of its own in M0
    ("s_add_u32 s2, s2, 1", "s_mov_b32 m0, s9", "M0 is used outside"),
    ("s_add_u32 s2, s2, 1", "ds_gws_init v0 gds", None),
    # the load right behind its M0, without the wait state between the two
    ("s_mov_b32 m0, s3\n\ts_nop 0\n", "s_mov_b32 m0, s3\n", "no wait state"),
    # spill space in a kernel with such loads
    (".amdhsa_private_segment_fixed_size 0", ".amdhsa_private_segment_fixed_size 64", "bytes of scratch"),
    # a register load that no hand-placed wait follows
    ("s_waitcnt vmcnt(1)", "s_nop 0", "no hand-placed s_waitcnt"),
])
def test_each_break_is_named(old, new, message):
    assert old in GOOD
    found = isa_check.violations(GOOD.replace(old, new, 1), "x.hip")
    if message is None:
        assert found == []      # an instruction that does not touch M0 or the registers is no break
    else:
        assert any(message in v for v in found), found
        assert all(v.startswith("x.hip:") for v in found)


def test_requests_with_a_scalar_base_are_hand_loads_too():
    # `global_load_lds_dwordx4 vOFFSET, s[BASE]`: one vector register of lane offsets, the base in scalar registers
    scalar = GOOD.replace("global_load_lds_dwordx4 v[2:3], off", "global_load_lds_dwordx4 v14, s[8:9]", 1)
    assert scalar != GOOD and isa_check.violations(scalar) == []
    broken = scalar.replace("s_add_u32 s2, s2, 1", "global_load_dword v11, v[2:3], off", 1)
    assert any("hand-counted wait" in v for v in isa_check.violations(broken, "x.hip"))
    broken = scalar.replace("s_add_u32 s2, s2, 1", "s_mov_b32 m0, s9", 1)
    assert any("M0 is used outside" in v for v in isa_check.violations(broken, "x.hip"))


def test_a_store_may_stand_behind_a_request_into_lds_but_not_behind_a_register_load():
    # vmcnt counts stores too and everything retires in order: a store among the later operations only
    # lengthens the wait for a request into LDS.  Behind a load into registers it stays a break (the
    # scan cannot tell which of the two waits the author counted).
    store = "global_store_dwordx4 v[20:21], v[22:25], off"
    lds_only = GOOD.replace("global_load_dwordx2 v[4:5], v[2:3], off", "s_nop 0", 1)
    assert isa_check.violations(lds_only.replace("s_add_u32 s2, s2, 1", store, 1)) == []
    both = isa_check.violations(GOOD.replace("s_add_u32 s2, s2, 1", store, 1), "x.hip")
    assert any("hand-counted wait" in v for v in both), both
    # a load of the compiler's behind the same request is still named
    load = lds_only.replace("s_add_u32 s2, s2, 1", "global_load_dword v11, v[2:3], off", 1)
    assert any("hand-counted wait" in v for v in isa_check.violations(load, "x.hip"))


COUNTED = """
_Z4rowsv:
	global_load_lds_dwordx4 v[2:3], off
	global_load_lds_dwordx4 v[4:5], off
	global_load_dwordx4 v[8:11], v[6:7], off
	global_load_dwordx4 v[12:15], v[6:7], off offset:16
	;;#ASMSTART
	s_waitcnt vmcnt(2)
	;;#ASMEND
	ds_read_b128 v[20:23], v1
	s_endpgm
.Lfunc_end0:
"""


def test_the_compilers_loads_behind_a_counted_lds_load_are_counted():
    assert isa_check.counted_violations(COUNTED) == []
    # one of them moved ahead of the LDS-direct loads: two outstanding loads could include the awaited one
    load = "\tglobal_load_dwordx4 v[12:15], v[6:7], off offset:16\n"
    moved = COUNTED.replace(load, "", 1).replace("_Z4rowsv:\n", "_Z4rowsv:\n" + load, 1)
    assert any("1 register loads follow" in v for v in isa_check.counted_violations(moved, "x.hip"))
    # both of them, in a kernel whose second run of LDS-direct loads is in order: the wait has closed the first run
    first = COUNTED[COUNTED.index("\tglobal_load_lds"):COUNTED.index("\ts_endpgm")]
    loads = "".join(line + "\n" for line in first.splitlines() if "global_load_dwordx4" in line)
    two_runs = COUNTED.replace(first, first + first, 1)
    assert isa_check.counted_violations(two_runs) == []
    ahead = COUNTED.replace(first, loads + first.replace(loads, "", 1) + first, 1)
    found = isa_check.counted_violations(ahead, "x.hip")
    assert len(found) == 1 and "0 register loads follow" in found[0], found
    unwaited = COUNTED.replace("s_waitcnt vmcnt(2)", "s_nop 0", 1)
    assert any("without a hand-placed wait" in v for v in isa_check.counted_violations(unwaited, "x.hip"))


LOOP = """
_Z4loopv:
	s_mov_b32 s0, 0
.LBB0_1:
	;;#ASMSTART
	s_waitcnt vmcnt(2)
	;;#ASMEND
	ds_read_b128 v[20:23], v1
	;;#ASMSTART
	s_mov_b32 m0, s3
	s_nop 0
	global_load_lds_dwordx4 v2, s[8:9]
	;;#ASMEND
	;;#ASMSTART
	s_mov_b32 m0, s4
	s_nop 0
	global_load_lds_dwordx4 v3, s[8:9]
	;;#ASMEND
	global_load_dwordx4 v[8:11], v[6:7], off
	global_load_dwordx4 v[12:15], v[6:7], off offset:16
	s_cbranch_scc1 .LBB0_1
	;;#ASMSTART
	s_waitcnt vmcnt(0)
	;;#ASMEND
	s_endpgm
.Lfunc_end0:
	.amdhsa_kernel _Z4loopv
		.amdhsa_private_segment_fixed_size 0
	.end_amdhsa_kernel
"""
HAND = isa_check.HAND_ISSUED_SOURCES[0]


@pytest.mark.parametrize("source", ["x.hip", HAND])
def test_counted_loads_are_counted_along_a_branch_back_over_them(source):
    assert isa_check.counted_violations(LOOP, source) == []
    # one register load less on the way round; on the way out nothing is left outstanding
    load = "\tglobal_load_dwordx4 v[12:15], v[6:7], off offset:16\n"
    found = isa_check.counted_violations(LOOP.replace(load, "", 1), source)
    assert any("1 register loads follow" in v and "allows 2" in v for v in found), found
    # the same load behind the branch is not on the way round either
    found = isa_check.counted_violations(LOOP.replace(load, "", 1).replace("s_cbranch_scc1 .LBB0_1\n", "s_cbranch_scc1 .LBB0_1\n" + load, 1),
                                         source)
    assert any("1 register loads follow" in v and "allows 2" in v for v in found), found


def test_the_compilers_lds_loads_find_their_own_m0():
    mixed = COUNTED.replace("_Z4rowsv:\n", "_Z4rowsv:\n\t;;#ASMSTART\n\ts_mov_b32 m0, s4\n\t;;#ASMEND\n"
                            "\ts_mov_b32 m0, s5\n\ts_nop 0\n\tbuffer_load_dwordx4 v1, s[0:3], 0 offen lds\n")
    assert isa_check.counted_violations(mixed) == []
    found = isa_check.counted_violations(mixed.replace("\ts_mov_b32 m0, s5\n", ""), "x.hip")
    assert found and "finds M0 as an asm statement left it" in found[0], found
    found = isa_check.counted_violations(mixed.replace("\ts_nop 0\n", ""), "x.hip")
    assert len(found) == 1 and "no wait state" in found[0], found
    # M0 is read, or written for something that is no load into LDS of the compiler's
    for line in ("\ts_mov_b32 s9, m0\n", "\ts_add_u32 m0, m0, s9\n", "\tv_movrels_b32_e32 v1, m0\n"):
        found = isa_check.counted_violations(mixed.replace("\ts_mov_b32 m0, s5\n", line + "\ts_mov_b32 m0, s5\n"), "x.hip")
        assert len(found) == 1 and "M0 is used outside" in found[0], found
    found = isa_check.counted_violations(mixed.replace("\tds_read_b128", "\ts_mov_b32 m0, s6\n\tds_read_b128"), "x.hip")
    assert len(found) == 1 and "M0 is used outside" in found[0], found


def test_hand_issued_counted_loads_need_a_wait_behind_them():
    end = LOOP[LOOP.index("\tglobal_load_dwordx4 v[8:11]"):LOOP.index("\ts_endpgm")]
    straight = LOOP.replace(end, "", 1)     # a run with nothing behind it but the function's end
    found = isa_check.counted_violations(straight, HAND)
    assert any("no hand-placed wait follows" in v for v in found), found
    # where the compiler issues the runs, such a one is held to the strictest wait of the kernel, and so is one whose next wait is laxer
    assert any("0 register loads follow" in v for v in isa_check.counted_violations(straight, "x.hip"))
    last = LOOP.replace("\ts_cbranch_scc1 .LBB0_1\n", "", 1)
    last = last.replace("\tglobal_load_dwordx4 v[12:15], v[6:7], off offset:16\n", "", 1)    # 1 behind, then vmcnt(0)
    assert isa_check.counted_violations(last, HAND) == []
    assert any("1 register loads follow" in v for v in isa_check.counted_violations(last, "x.hip"))


def test_hand_issued_counted_loads_keep_m0_and_have_no_scratch():
    assert isa_check.m0_violations(LOOP, HAND) == []
    broken = LOOP.replace("s_mov_b32 s0, 0", "s_mov_b32 m0, s0", 1)
    assert any("M0 is used outside" in v for v in isa_check.m0_violations(broken, HAND))
    broken = LOOP.replace("fixed_size 0", "fixed_size 16", 1)
    assert any("bytes of scratch" in v for v in isa_check.m0_violations(broken, HAND))
    # what else is in flight is not this check's business
    assert isa_check.violations(LOOP, HAND) != []


def test_the_release_is_read_from_hipcc_version_text():
    assert isa_check.hipcc_release("HIP version: 7.2.26015-fc0010cf6a\nAMD clang version 22") == "7.2.26015"
    assert isa_check.hipcc_release("nothing") == ""


def test_the_built_library_came_through_the_check():
    # the assembly texts the last build checked lie beside its objects; they pass, and they
    # do contain the statements the check is about
    texts = [os.path.join(build.OBJ_DIR, os.path.splitext(s)[0] + ".s") for s in isa_check.CHECKED_SOURCES]
    if not all(os.path.exists(t) for t in texts):
        pytest.skip("no build in this tree yet")
    for path in texts:
        with open(path) as f:
            asm = f.read()
        assert isa_check.violations(asm, os.path.basename(path)) == []
        assert "global_load_lds_dwordx4" in asm
    for source in isa_check.COUNTED_SOURCES:
        with open(os.path.join(build.OBJ_DIR, os.path.splitext(source)[0] + ".s")) as f:
            asm = f.read()
        assert isa_check.counted_violations(asm, source) == []
        assert "global_load_lds_dwordx4" in asm
        if source in isa_check.HAND_ISSUED_SOURCES:
            assert isa_check.m0_violations(asm, source) == []
