"""The build's check of the register-resident kernels' device assembly (_build.check_bank), on listings with and without
the faults it looks for. The build itself runs it on every size class."""
import pytest

from decaes_amd import _build

OK = """
nnls:
	v_add_f64 v[94:95], v[2:3], v[4:5]
	v_mov_b32_e32 v1, v0
	;;#ASMSTART
	s_nop 1
	v_fmac_f64_dpp v[96:97], v[94:95], v[4:5] row_newbcast:0 row_mask:0xf bank_mask:0xf
	v_fmac_f64_dpp v[254:255], v[94:95], v[4:5] row_newbcast:1 row_mask:0xf bank_mask:0xf
	;;#ASMEND
	.set nnls.num_vgpr, 96 ; v200
	ds_write_b64 v1, v[94:95]
"""


def test_accepts_the_bank_in_inline_assembly_only():
    _build.check_bank(OK, 80)


@pytest.mark.parametrize("line", ["v_mov_b32_e32 v96, v0", "global_load_dwordx4 v[93:96], v[2:3], off",
                                  "v_add_f64 v[2:3], v[4:5], |v[254:255]|", "scratch_store_dword off, v255, s32"])
def test_refuses_a_compiler_use_of_the_bank(line):
    with pytest.raises(RuntimeError, match="solver's registers"):
        _build.check_bank(OK + "\t" + line + "\n", 80)
    _build.check_bank((OK + "\t" + line + "\n").replace("v96", "v95").replace("93:96", "92:95").replace("254:255", "94:95")
                      .replace("v255", "v95"), 80)


@pytest.mark.parametrize("between,ok", [("", False), ("\ts_nop 0\n", False), ("\tv_mov_b32_e32 v9, v8\n", False),
                                        ("\ts_nop 1\n", True), ("\ts_nop 0\n\ts_mov_b32 s0, 0\n", True)])
def test_refuses_a_dpp_read_right_after_its_source_is_written(between, ok):
    asm = ("\tv_mul_f64 v[6:7], v[2:3], v[4:5]\n" + between + "\t;;#ASMSTART\n"
           "\tv_fmac_f64_dpp v[96:97], v[6:7], v[4:5] row_newbcast:0 row_mask:0xf bank_mask:0xf\n\t;;#ASMEND\n")
    if ok:
        _build.check_bank(asm, 80)
    else:
        with pytest.raises(RuntimeError, match="too closely"):
            _build.check_bank(asm, 80)
