"""The library build's m0 guard (triton_llm/_build.py check_m0): kernels
that issue the inline-asm LDS-DMA, which writes m0, must contain no
compiler-generated m0 use.  Checked here on small assembly listings; the
build runs it on every device object."""

import pytest

from triton_llm import _build

DMA = """\t;;#ASMSTART
\ts_mov_b32 m0, s4
\tbuffer_load_dwordx4 v1, s[8:11], 0 offen lds
\t;;#ASMEND
"""


def listing(name, body):
    return f"\t.type\t{name},@function\n{name}:\n{body}\ts_endpgm\n.Lfunc_end0:\n"


def test_dma_kernel_without_compiler_m0_passes():
    text = listing("k_dma", "\tv_mov_b32 v0, 0\n" + DMA + "\ts_waitcnt vmcnt(0)\n")
    assert _build.check_m0(text, "t.hip") == 1


@pytest.mark.parametrize("use", ["\ts_mov_b32 m0, s2\n", "\tv_movrels_b32 v0, v1\n",
                                 "\tbuffer_load_dword v2, s[0:3], 0 offen lds\n"])
def test_compiler_m0_use_in_a_dma_kernel_fails(use):
    # in another basic block of the same kernel, after the asm
    text = listing("k_bad", DMA + ".LBB0_2:\n" + use)
    with pytest.raises(RuntimeError, match="k_bad"):
        _build.check_m0(text, "t.hip")


def test_m0_use_in_a_kernel_without_the_dma_is_allowed():
    text = listing("k_dma", DMA) + listing("k_other", "\ts_mov_b32 m0, -1\n\tds_read_b32 v0, v1\n")
    assert _build.check_m0(text, "t.hip") == 1


MFMA = "\t;;#ASMSTART\n\tv_mfma_f32_16x16x32_f16 a[0:3], v[4:7], v[8:11], a[0:3]\n\t;;#ASMEND\n"


def test_spaced_asm_mfma_passes():
    text = listing("k_mfma", "\tv_mov_b32_e32 v4, v1\n\ts_nop 1\n" + MFMA + "\ts_nop 10\n\tv_accvgpr_read_b32 v0, a1\n")
    assert _build.check_mfma_asm(text, "t.hip") == 1
    assert _build.check_mfma_asm(listing("k_other", "\tv_mfma_f32_16x16x32_f16 a[0:3], v[4:7], v[8:11], 0\n"), "t.hip") == 0


@pytest.mark.parametrize("body", [
    "\tv_mov_b32_e32 v9, v1\n\ts_nop 0\n" + MFMA,                          # operand written one state before
    "\tv_accvgpr_write_b32 a2, v1\n" + MFMA,                               # accumulator likewise
    MFMA + "\ts_nop 9\n\tv_accvgpr_read_b32 v0, a3\n",                     # result read one state early
    MFMA + "\tv_accvgpr_write_b32 a0, v1\n",                               # result overwritten
    ".LBB0_1:\n\tv_accvgpr_read_b32 v0, a3\n\ts_nop 10\n" + MFMA + "\ts_cbranch_scc0 .LBB0_1\n",  # around a loop
])
def test_asm_mfma_without_its_wait_states_fails(body):
    with pytest.raises(RuntimeError, match="k_bad"):
        _build.check_mfma_asm(listing("k_bad", body), "t.hip")
