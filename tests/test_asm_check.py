"""The build's assembly check (tcc_spmm_amd/asm_check.py) on small hand-written listings, and on
the kernel source as built here."""
import re

import pytest

from tcc_spmm_amd import asm_check, build

HEAD = "_ZN4test10TestKernelEv:\n"
TAIL = "\ts_endpgm\n.Lfunc_end0:\n"


def _listing(body: str) -> str:
    return HEAD + body + TAIL


def test_early_read_is_flagged():
    problems = asm_check.check(_listing(
        "\tv_mfma_f32_32x32x8_f16 v[0:15], v[16:17], v[18:19], v[0:15]\n"
        "\ts_nop 3\n"
        "\tv_mov_b32_e32 v20, v3\n"))
    assert len(problems) == 1 and "4 wait states" in problems[0]  # s_nop 3 = 4


def test_padded_read_and_accumulator_chain_pass():
    assert asm_check.check(_listing(
        "\tv_mfma_f32_32x32x8_f16 v[0:15], v[16:17], v[18:19], v[0:15]\n"
        "\tv_mfma_f32_32x32x8_f16 v[0:15], v[20:21], v[18:19], v[0:15]\n"
        "\ts_nop 7\n\ts_nop 7\n\ts_nop 1\n"
        "\tv_mov_b32_e32 v20, v3\n")) == []


def test_read_on_a_branch_path_is_flagged():
    problems = asm_check.check(_listing(
        "\tv_mfma_f32_32x32x8_f16 v[0:15], v[16:17], v[18:19], v[0:15]\n"
        "\ts_cbranch_scc1 .LBB0_2\n"
        "\ts_nop 7\n\ts_nop 7\n\ts_nop 7\n"
        ".LBB0_2:\n"
        "\tglobal_store_dwordx4 v[30:31], v[0:3], off\n"))
    assert len(problems) == 1 and "global_store_dwordx4" in problems[0]


def test_overwritten_register_is_not_a_read_of_the_result():
    assert asm_check.check(_listing(
        "\tv_mfma_f32_32x32x8_f16 v[0:15], v[16:17], v[18:19], v[0:15]\n"
        "\tv_mov_b32_e32 v20, v40\n")) == []


def test_spill_is_flagged():
    problems = asm_check.check(_listing("\tscratch_store_dwordx4 off, v[4:7], off offset:16\n"))
    assert any("spills" in p for p in problems)


def _walk(between, wait="s_waitcnt vmcnt(4)", rows=2):
    """A loop like the panel walk's: other loads, a pair's X rows to LDS, the wait and the reads of the
    pair loaded one turn earlier."""
    row = "\tbuffer_load_dwordx4 v9, s[4:7], 0 offen lds\n"
    body = row * rows + ".LBB0_1:\n" + between + row * rows
    body += f"\t;;#ASMSTART\n\t{wait}\n" + "\tds_read_b32 v1, v2\n"
    return _listing(body + "\t;;#ASMEND\n\ts_cbranch_scc1 .LBB0_1\n")


LOAD = "\tbuffer_load_dword v3, v4, s[4:7], 0 offen\n"


def test_wait_that_covers_the_pair_passes():
    assert asm_check.check(_walk(LOAD * 2)) == []
    assert asm_check.check(_walk(LOAD * 5)) == []                        # stricter than it need be
    assert asm_check.check(_walk(LOAD, wait="s_waitcnt vmcnt(3)")) == []
    # loads drained on the way: nothing of the pair is outstanding
    assert asm_check.check(_walk(LOAD + "\ts_waitcnt vmcnt(0)\n")) == []
    assert asm_check.check(_walk(LOAD * 2).replace("lds\n", "offset:16\n")) == []  # no loads to LDS


def test_wait_one_instruction_short_is_flagged():
    """A load dropped, merged or sunk below the reads, a wait for fewer, and a row of the next pair that is
    loaded after the wait."""
    problems = asm_check.check(_walk(LOAD))
    assert len(problems) == 1 and "vmcnt(4)" in problems[0]
    assert len(asm_check.check(_walk(LOAD * 2, wait="s_waitcnt vmcnt(5)"))) == 1
    assert asm_check.check(_walk(LOAD * 3, rows=1)) == []
    assert len(asm_check.check(_walk(LOAD * 2, rows=1))) == 1


def test_wait_on_a_path_that_skips_a_load_is_flagged():
    assert len(asm_check.check(_walk("\ts_cbranch_vccnz .LBB0_2\n" + LOAD + ".LBB0_2:\n" + LOAD))) == 1


def test_wide_kernel_counts_four_rows_a_pair():
    listing = _walk(LOAD * 2, wait="s_waitcnt vmcnt(6)", rows=4)
    assert len(asm_check.check(listing)) == 1
    assert asm_check.check(listing.replace("10TestKernelEv", "13TestKernel256Ev")) == []


def test_operand_reads_without_a_wait_are_flagged():
    assert len(asm_check.check(_walk(LOAD * 2, wait="s_nop 0"))) == 1


def test_address_of_a_load_to_lds_is_a_read():
    problems = asm_check.check(_listing(
        "\tv_mfma_f32_32x32x8_f16 v[0:15], v[16:17], v[18:19], v[0:15]\n"
        "\tbuffer_load_dwordx4 v3, s[4:7], 0 offen lds\n"))
    assert len(problems) == 1 and "lds" in problems[0]


@pytest.fixture(scope="module")
def listing():
    """The assembly of the SpMM kernels, compiled and checked as in every build."""
    build.check_kernel_asm()
    return (build.BUILD / "spmm-gfx950.s").read_text()


def test_kernel_source_passes(listing):
    """The shipped SpMM kernels compile to clean assembly (this is also part of every build)."""
    assert asm_check.check(listing) == []
    # The waits of the panel walk are seen: without the pair's last value load (the last indexed load
    # ahead of its X rows) every kernel that loads X rows to LDS, the buffer-addressed ones, is refused.
    lines, dropped = [], None
    for line in listing.split("\n"):
        if line.rstrip().endswith(" lds") and dropped is not None:
            del lines[dropped]
            dropped = None
        if line.startswith("\tbuffer_load_dword ") and line.rstrip().endswith("idxen"):
            dropped = len(lines)
        lines.append(line)
    short = [p for p in asm_check.check("\n".join(lines)) if "load to LDS" in p]
    kernels = {p.split(":")[0] for p in short}
    assert len(kernels) == 8 and all("ILj0E" in k for k in kernels)


def test_wave_slots_are_those_of_the_compiled_instances(listing):
    """The launch prices a plan against CUs x 4 SIMDs x the waves per SIMD it takes an instance to run;
    the compiled instances run that many."""
    occupancy = {}
    for m in re.finditer(r"^_ZN\S*spmmInt8Kernel(\d+)ILj(\d)E[^\s:]*:", listing, re.M):
        waves = int(re.search(r"^; Occupancy: (\d+)", listing[m.end():], re.M).group(1))
        occupancy.setdefault((int(m.group(1)), int(m.group(2))), set()).add(waves)
    source = (build.CSRC / "kernel" / "spmm.hip").read_text()
    rule = re.search(r"constexpr unsigned wavesPerSimd\(.*?return (.*?);", source, re.S).group(1)
    assert rule == "features == 256 ? 2 : addr == kBuffer ? 4 : 3"
    assert "waveSlots(Features, addr)" in source
    want = {(f, a): {2 if f == 256 else 4 if a == 0 else 3} for f in (128, 256) for a in (0, 1, 2)}
    assert occupancy == want
