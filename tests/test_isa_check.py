"""The check of the built gfx950 code: planted sequences, and the library."""
import pytest

from mbsolve_amd import capi, isa_check

FMAC = "v_fmac_f64_dpp v[0:1], v[2:3], v[4:5] row_newbcast:3 row_mask:0xf " \
    "bank_mask:0xf"


def _listing(lines, name="some_kernel"):
    """llvm-objdump's form, four bytes per instruction; 'to N' is a branch to
    line N."""
    out = ["0000000000001000 <%s>:" % name]
    for k, text in enumerate(lines):
        op = text.split()[0]
        if " to " in text:
            off = (int(text.split()[-1]) - k - 1) % 65536
            text = "%s %d" % (op, off)
        out.append("\t%s // %012X: 00000000" % (text, 0x1000 + 4 * k))
    return "\n".join(out) + "\n"


@pytest.mark.parametrize("lines,bad", [
    (["v_mov_b32_e32 v3, v9", FMAC], True),
    (["v_mov_b32_e32 v3, v9", "s_nop 0", FMAC], True),
    (["v_mov_b32_e32 v3, v9", "s_nop 1", FMAC], False),
    (["v_mov_b32_e32 v3, v9", "s_mov_b32 s0, 0", "s_mov_b32 s1, 0", FMAC],
     False),
    (["v_accvgpr_read_b32 v2, a7", "s_waitcnt vmcnt(0)", FMAC], True),
    # the operands that DPP does not read are interlocked
    (["v_add_f64 v[4:5], v[6:7], v[8:9]", FMAC], False),
    (["v_mul_f64 v[0:1], v[6:7], v[8:9]", FMAC], False),
    (["v_rcp_f64_e32 v[4:5], v[6:7]", FMAC], True),
    (["v_rcp_f64_e32 v[4:5], v[6:7]", "s_nop 0", FMAC], False),
    (["v_cmpx_lt_f64_e32 v[6:7], v[8:9]", "s_nop 3", FMAC], True),
    (["v_cmpx_lt_f64_e32 v[6:7], v[8:9]", "s_nop 4", FMAC], False),
    (["v_mfma_f32_16x16x32_f16 v[4:7], v[8:11], v[12:15], v[4:7]",
      "s_nop 15", FMAC], True),
    # by the way of a branch, forward and backward
    (["v_mov_b32_e32 v3, v9", "s_cbranch_scc0 to 6", "s_nop 7", "s_nop 7",
      "s_nop 7", "s_endpgm", FMAC], True),
    (["s_nop 7", FMAC, "s_nop 7", "v_mov_b32_e32 v2, v9",
      "s_cbranch_scc1 to 1", "s_endpgm"], True),
    (["s_branch to 3", "v_mov_b32_e32 v2, v9", "s_endpgm", FMAC], False),
    (["v_mov_b32_e32 v3, v9", "s_endpgm", FMAC], False),
])
def test_planted_sequences(lines, bad):
    count, found = isa_check.hazards(_listing(["s_nop 15", "s_nop 15"]) +
                                     _listing(lines))
    assert count == 1
    assert bool(found) == bad, found


def test_function_entry_counts_as_unknown():
    assert isa_check.hazards(_listing([FMAC], "helper"))[1]
    assert not isa_check.hazards(_listing(["s_nop 4", FMAC], "helper"))[1]


def test_library_keeps_the_wait_states():
    assert isa_check.check(capi.LIB_PATH) > 1000
