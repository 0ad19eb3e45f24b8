"""The build's scan of inline-asm MFMAs (raftinfer_amd/asm_check.py) on small
listings whose answer is fixed by counting wait states, and on the built
prefill kernel itself."""
import pathlib

from raftinfer_amd import asm_check
from raftinfer_amd.asm_check import RESULT_WAIT_STATES, asm_mfma_hazards

MFMA = """\t;;#ASMSTART
\ts_nop 1
\tv_mfma_f32_32x32x16_bf16 a[16:31], v[30:33], v[6:9], a[16:31]
\t;;#ASMEND
"""


def test_copy_right_after_an_asm_mfma_is_flagged():
    text = MFMA + "\tv_accvgpr_mov_b32 a2, a17\n"
    hazards = asm_mfma_hazards(text)
    assert len(hazards) == 1 and "a[16:31]" in hazards[0] and "after 0 wait states" in hazards[0]


def test_reads_after_the_drain_or_of_other_registers_pass():
    drained = MFMA + "\ts_nop 7\n\ts_nop 7\n\ts_nop 3\n\tv_accvgpr_read_b32 v0, a16\n"
    assert asm_mfma_hazards(drained) == []
    other = MFMA + "\tv_accvgpr_read_b32 v0, a32\n\tv_accvgpr_mov_b32 a1, a15\n"
    assert asm_mfma_hazards(other) == []


def test_wait_states_are_counted_exactly():
    # s_nop n gives n + 1 wait states; one short of the latency is flagged, the latency is not
    short = MFMA + "\ts_nop 7\n" * 2 + f"\ts_nop {RESULT_WAIT_STATES - 16 - 2}\n" + "\tv_add_f32 v1, a20, v2\n"
    assert len(asm_mfma_hazards(short)) == 1
    enough = MFMA + "\ts_nop 7\n" * 2 + f"\ts_nop {RESULT_WAIT_STATES - 16 - 1}\n" + "\tv_add_f32 v1, a20, v2\n"
    assert asm_mfma_hazards(enough) == []


def test_compiler_mfmas_and_mfma_chains_are_not_flagged():
    # a compiler-placed MFMA (outside ASMSTART/ASMEND) is the compiler's own business, and an
    # accumulator chain is checked by the hardware
    text = "\tv_mfma_f32_32x32x16_bf16 a[0:15], v[4:7], v[8:11], 0\n\tv_accvgpr_read_b32 v0, a0\n"
    text += MFMA + MFMA
    assert asm_mfma_hazards(text) == []


def test_vector_results_operand_writes_and_owned_registers():
    mfma = MFMA.replace("\ts_nop 1\n", "").replace("a[16:31]", "v[40:55]")
    for line in ("\tv_mov_b32_e32 v1, v41\n", "\tv_mov_b32_e32 v55, v1\n", "\tds_write_b32 v1, v50\n"):
        assert len(asm_mfma_hazards(mfma + line)) == 1, line
        assert asm_mfma_hazards(mfma + "\ts_nop 7\n" * 3 + line) == [], line
    # an operand written by the vector unit right before, then two wait states before
    write = "\tv_add_f32_e32 v32, v1, v2\n"
    assert len(asm_mfma_hazards(write + "\ts_nop 0\n" + mfma)) == 1
    assert asm_mfma_hazards(write + "\ts_nop 1\n" + mfma) == []
    # ... also the accumulator that goes in, and both registers of a swap
    for line in ("\tv_accvgpr_write_b32 a20, v9\n", "\tv_permlane32_swap_b32_e32 v1, v31\n",
                 "\tv_permlane32_swap_b32_e32 v9, v1\n", "\tv_swap_b32 v1, v7\n"):
        agpr = MFMA.replace("\ts_nop 1\n", "")
        assert len(asm_mfma_hazards(line + agpr)) == 1, line
        assert asm_mfma_hazards(line + "\ts_nop 1\n" + agpr) == [], line
    for line in ("\tv_permlane32_swap_b32_e32 v1, v41\n", "\tv_permlane16_swap_b32_e32 v41, v1\n"):
        assert len(asm_mfma_hazards(mfma + line)) == 1, line
    # registers named in hexadecimal, and the rule for kernels that own the accumulation registers
    assert len(asm_mfma_hazards(MFMA.replace("a[16:31]", "a[0x80:0x8f]") + "\tv_accvgpr_read_b32 v0, a[0x81]\n")) == 1
    spill = "\tv_accvgpr_write_b32 a3, v9\n"
    assert asm_mfma_hazards(spill) == []
    assert len(asm_mfma_hazards(spill, owned_agprs=True)) == 1
    assert asm_mfma_hazards("\t;;#ASMSTART\n" + spill + "\t;;#ASMEND\n", owned_agprs=True) == []


def test_built_prefill_kernel_has_no_hazard():
    s = pathlib.Path(asm_check.__file__).resolve().parent / "_build" / "attention_prefill_mfma.hip.s"
    if not s.exists():
        import pytest
        pytest.skip("the library has not been built here")
    assert asm_mfma_hazards(s.read_text()) == []
    wide = s.with_name("attention_prefill_wide.hip.s")
    assert asm_mfma_hazards(wide.read_text(), owned_agprs=True) == []
