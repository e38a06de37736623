"""The assembly audit accepts the instructions it lists and refuses any
other scalar or memory instruction (made-up names here)."""

import pytest

from sigcomp_amd import isa_audit

LISTED = """
	s_load_dwordx4 s[0:3], s[4:5], 0x0
	s_add_u32 s0, s0, s1
	s_mul_hi_i32 s0, s0, s1
	s_and_saveexec_b64 s[0:1], vcc
	s_cmp_lg_u64 s[0:1], 0
	s_cbranch_scc1 .LBB0_1
	s_waitcnt vmcnt(0)
	v_add_u32_e32 v0, v1, v2
	global_store_dwordx4 v[0:1], v[2:5], off
	buffer_load_dwordx4 v[0:3], v4, s[0:3], 0 offen
	ds_read2st64_b32 v[0:1], v2 offset1:1
	ds_write_b8 v0, v1
	s_endpgm
"""


def test_listed_instructions_pass():
    isa_audit.check(LISTED)


@pytest.mark.parametrize("name", ["s_keep_dword", "s_load_dwordx4_back", "s_buffer_keep_dwordx2", "s_add_u32_keep",
                                  "global_keep_dword", "flat_load_dword", "ds_keep_b32", "buffer_keep_dwordx2"])
@pytest.mark.parametrize("operands", [" s[0:1], s2", ""])
def test_any_other_is_refused(name, operands):
    with pytest.raises(RuntimeError, match=f"'{name}'"):
        isa_audit.check(LISTED + f"\t{name}{operands}\n")
