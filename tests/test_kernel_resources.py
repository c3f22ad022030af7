"""Register budgets that are part of a kernel's design, held to the build's own resource report.

The 8-bit attention kernels' register budget is part of their design: one wave per SIMD with
the whole register file, 128 accumulators in ordinary registers, the q terms in the accumulation
registers (rivoli_amd/csrc/mla_attend_f8.hpp). A compiler or source change that makes them spill
still gives right answers, only several times slower, so the build's own resource report is held
to "no scratch memory" here. The scored block selection keeps a row's keys in registers and its
phases must not share per-element lane masks: 32 of them do not fit the scalar registers, and
when they spilled (to lanes of a vector register, a write and a read each) a quarter of the
kernel's vector instructions were spill traffic. Compiles one file per test; needs hipcc, no
GPU."""
import functools
import os
import re
import shutil
import subprocess

import pytest

from rivoli_amd import build
from tests import wait_states


def test_the_build_compiles_with_the_flags_that_these_tests_compile_with(monkeypatch):
    """The tests below ask build.compile_command for their flags: a flag that only the build had would make another program of
    what is shipped than of what they look at."""
    ran = []

    def run(cmd, **_):
        ran.append(cmd)
        return subprocess.CompletedProcess(cmd, 0, "", "")

    monkeypatch.setattr(build.subprocess, "run", run)
    monkeypatch.setattr(build, "check_resources", lambda k, report: None)
    build.build_kernels()
    compiles = [cmd for cmd in ran if "-c" in cmd]
    assert sorted(os.path.basename(cmd[cmd.index("-c") + 1]) for cmd in compiles) == sorted(build.KERNELS)
    for cmd in compiles:
        flags = cmd[:cmd.index("-c")]
        own = build.compile_command(os.path.basename(cmd[cmd.index("-c") + 1]))
        assert flags[:len(own)] == own and set(flags[len(own):]) <= {"-Rpass-analysis=kernel-resource-usage"}


@pytest.mark.skipif(shutil.which(build.hipcc()) is None, reason="hipcc not found")
def test_eight_bit_attention_kernels_do_not_spill(tmp_path):
    src = os.path.join(build.CSRC, "mla_attend.hip")
    cmd = build.compile_command("mla_attend.hip") + \
          ["-Rpass-analysis=kernel-resource-usage", "-c", src, "-o", str(tmp_path / "m.o")]
    res = subprocess.run(cmd, capture_output=True, text=True)
    assert res.returncode == 0, res.stderr[-2000:]
    # remarks come in blocks: "Function Name: <mangled>" followed by that kernel's figures
    blocks = re.split(r"remark: Function Name: ", res.stderr)[1:]
    seen = 0
    for b in blocks:
        name = b.split()[0]
        if "mla_attend_paged_kernel" not in name or not name.endswith("Lb1EEEvNS_10AttendArgsE"):
            continue  # the last template argument (true) marks the 8-bit kernels
        seen += 1
        scratch = int(re.search(r"ScratchSize \[bytes/lane\]: (\d+)", b).group(1))
        occupancy = int(re.search(r"Occupancy \[waves/SIMD\]: (\d+)", b).group(1))
        lds = int(re.search(r"LDS Size \[bytes/block\]: (\d+)", b).group(1))
        assert scratch == 0, f"{name} spills {scratch} bytes per lane"
        assert occupancy == 1, name
        assert lds <= 160 * 1024, name
    assert seen == 4, f"expected the dense and row-list kernels of both 8-bit modes, saw {seen}"


@functools.lru_cache(maxsize=None)
def _compiled(src_name):
    """The file's resource report and its listing."""
    cmd = build.compile_command(src_name) + \
          ["-Rpass-analysis=kernel-resource-usage", "--cuda-device-only", "-S", os.path.join(build.CSRC, src_name), "-o", "-"]
    res = subprocess.run(cmd, capture_output=True, text=True)
    assert res.returncode == 0, res.stderr[-2000:]
    return res.stderr, res.stdout


def _resource_blocks(src_name):
    return re.split(r"remark: Function Name: ", _compiled(src_name)[0])[1:]


@pytest.mark.skipif(shutil.which(build.hipcc()) is None, reason="hipcc not found")
def test_block_selection_keeps_its_masks_out_of_memory():
    seen = 0
    for b in _resource_blocks("index_topk.hip"):
        name = b.split()[0]
        if "block_select_bisect_kernel" not in name:
            continue
        seen += 1
        assert int(re.search(r"SGPRs Spill: (\d+)", b).group(1)) == 0, name
        assert int(re.search(r"VGPRs Spill: (\d+)", b).group(1)) == 0, name
        assert int(re.search(r"ScratchSize \[bytes/lane\]: (\d+)", b).group(1)) == 0, name
        assert int(re.search(r"Occupancy \[waves/SIMD\]: (\d+)", b).group(1)) == 8, name
    assert seen == 6, f"expected the six widths of the register form, saw {seen}"


@pytest.mark.skipif(shutil.which(build.hipcc()) is None, reason="hipcc not found")
def test_block_scorer_keeps_its_row_and_both_chunk_buffers_in_registers():
    """The block scorer holds a 128-value row per lane and two 32-value chunks of the query in
    scalar registers; a spill of either turns its two instructions per term into many."""
    seen = 0
    for b in _resource_blocks("block_index.hip"):
        name = b.split()[0]
        if "index_score_blocks_128" not in name:
            continue
        seen += 1
        if "split" not in name:   # the decode kernel is bound by latency, not by issue
            assert int(re.search(r"SGPRs Spill: (\d+)", b).group(1)) == 0, name
        assert int(re.search(r"VGPRs Spill: (\d+)", b).group(1)) == 0, name
        assert int(re.search(r"ScratchSize \[bytes/lane\]: (\d+)", b).group(1)) == 0, name
        assert int(re.search(r"Occupancy \[waves/SIMD\]: (\d+)", b).group(1)) >= 3, name
    assert seen == 2


@pytest.mark.skipif(shutil.which(build.hipcc()) is None, reason="hipcc not found")
def test_kernels_of_16_heads_a_workgroup_do_not_spill():
    """One wave per SIMD with the whole register file, transfers into LDS ordered by hand
    (rivoli_amd/csrc/mla_attend_heads16.hpp): dense and listed, in each of the bf16 modes."""
    seen = 0
    for b in _resource_blocks("mla_attend.hip"):
        name = b.split()[0]
        if "mla_attend_heads16_kernel" not in name:
            continue
        seen += 1
        assert int(re.search(r"VGPRs Spill: (\d+)", b).group(1)) == 0, name
        assert int(re.search(r"ScratchSize \[bytes/lane\]: (\d+)", b).group(1)) == 0, name
        assert int(re.search(r"Occupancy \[waves/SIMD\]: (\d+)", b).group(1)) == 1, name
        assert int(re.search(r"LDS Size \[bytes/block\]: (\d+)", b).group(1)) <= 160 * 1024, name
    assert seen == 6


@pytest.mark.skipif(shutil.which(build.hipcc()) is None, reason="hipcc not found")
def test_kernels_that_count_their_transfers_do_not_spill():
    """Eight waves on a tile of 64 tokens (rivoli_amd/csrc/mla_attend_few.hpp): a wave waits until six reads
    are left on their way, the next tile's; a spilled register's reload would be one more."""
    blocks = [b for b in _resource_blocks("mla_attend.hip") if "mla_attend_few_kernel" in b.split()[0]]
    assert len(blocks) == 7
    for b in blocks:
        name = b.split()[0]
        assert int(re.search(r"VGPRs Spill: (\d+)", b).group(1)) == 0, name
        assert int(re.search(r"ScratchSize \[bytes/lane\]: (\d+)", b).group(1)) == 0, name
        assert int(re.search(r"LDS Size \[bytes/block\]: (\d+)", b).group(1)) <= 160 * 1024, name


@pytest.mark.skipif(shutil.which(build.hipcc()) is None, reason="hipcc not found")
def test_the_block_scorers_matrix_kernels_and_the_few_row_selection_do_not_spill():
    """Two waves per SIMD of up to 255 registers in the many-query scorers (scalar registers do spill
    there, in the fold), three in the one-query scorers; a row's keys in registers and its masks
    out of memory in the few-row selection, as in the many-row one."""
    seen = []
    for src, part, waves in (("block_index.hip", "score_blocks_pair_kernel", 2),
                             ("block_index.hip", "score_blocks_codes_kernel", 2),
                             ("block_index.hip", "score_blocks_one_kernel", 3),
                             ("index_topk.hip", "block_select_few_kernel", 8),
                             ("index_topk.hip", "index_topk_few_kernel", 8)):
        for b in _resource_blocks(src):
            name = b.split()[0]
            if part not in name:
                continue
            seen.append(part)
            if src == "index_topk.hip":
                assert int(re.search(r"SGPRs Spill: (\d+)", b).group(1)) == 0, name
            assert int(re.search(r"VGPRs Spill: (\d+)", b).group(1)) == 0, name
            assert int(re.search(r"ScratchSize \[bytes/lane\]: (\d+)", b).group(1)) == 0, name
            assert int(re.search(r"Occupancy \[waves/SIMD\]: (\d+)", b).group(1)) >= waves, name
    assert len(seen) == 12 and seen.count("block_select_few_kernel") == seen.count("index_topk_few_kernel") == 4


def test_the_build_refuses_an_attention_object_that_spills():
    """build.check_resources is what build_kernels applies to mla_attend.hip's resource report:
    scratch memory or too much LDS in an 8-bit attention kernel, or in one of 16 heads a workgroup (a tile a
    wave, or eight waves on a tile) or of 32, raises instead of linking, and so does a report without one of these families."""
    figures = "    ScratchSize [bytes/lane]: 0\n    LDS Size [bytes/block]: 85632\n"
    head = "x.hip:1:1: remark: Function Name: _ZN2rk23mla_attend_paged_kernelILi2ELi2ELi0ELb0ELb1EEEvNS_10AttendArgsE\n"
    heads16 = "x.hip:1:1: remark: Function Name: _ZN2rk25mla_attend_heads16_kernelILi2ELi2ELi3EEEvNS_10AttendArgsE\n"
    few = "x.hip:1:1: remark: Function Name: _ZN2rk21mla_attend_few_kernelILi2ELi2ELi3EEEvNS_10AttendArgsE\n"
    wide = "x.hip:1:1: remark: Function Name: _ZN2rk22mla_attend_wide_kernelILi2ELi2ELi0EEEvNS_10AttendArgsE\n"
    families = [head + figures, heads16 + figures.replace("85632", "161328"), few + figures.replace("85632", "142912"),
                wide + figures.replace("85632", "162432")]
    fine = "".join(families)
    build.check_resources("mla_attend.hip", fine)
    build.check_resources("kv_gather.hip", "")                        # other files are not held to it
    for i, family in enumerate(families):
        others = "".join(families[:i] + families[i + 1:])
        for bad in (others, others + family.replace("lane]: 0", "lane]: 8"), others + re.sub(r"block\]: \d+", "block]: 163856", family)):
            with pytest.raises(RuntimeError):
                build.check_resources("mla_attend.hip", bad)
    for bad in ("", families[0], fine.replace("85632", "170000"), "lane]: 4".join(fine.rsplit("lane]: 0", 1))):
        with pytest.raises(RuntimeError):
            build.check_resources("mla_attend.hip", bad)


@pytest.mark.skipif(shutil.which(build.hipcc()) is None, reason="hipcc not found")
def test_attention_of_32_heads_a_workgroup_fits_its_registers_and_a_compute_units_lds():
    """Eight waves in half of the registers each, three tiles and four partial scores in nearly all of the LDS; both address modes of three modes."""
    blocks = [b for b in _resource_blocks("mla_attend.hip") if "mla_attend_wide_kernel" in b.split()[0]]
    assert len(blocks) == 6
    for b in blocks:
        assert int(re.search(r"ScratchSize \[bytes/lane\]: (\d+)", b).group(1)) == 0
        assert int(re.search(r"LDS Size \[bytes/block\]: (\d+)", b).group(1)) <= 160 * 1024


@pytest.mark.skipif(shutil.which(build.hipcc()) is None, reason="hipcc not found")
def test_list_attention_of_32_heads_a_wave_keeps_its_operands_apart(tmp_path):
    """Its score products are written as assembly, so the compiler does not see to their wait states:
    a vector instruction's result may be a matrix instruction's operand two instructions later at
    the earliest. Reads the listing; and no block with products may touch scratch memory, where the wait for
    it would be a wait for every row on its way."""
    out = tmp_path / "g.s"
    cmd = build.compile_command("gather_attn.hip") + \
          ["--cuda-device-only", "-S", os.path.join(build.CSRC, "gather_attn.hip"), "-o", str(out)]
    res = subprocess.run(cmd, capture_output=True, text=True)
    assert res.returncode == 0, res.stderr[-2000:]

    def registers(operand):
        m = re.fullmatch(r"v\[(\d+):(\d+)\]|v(\d+)", operand)
        if not m:
            return set()
        return {int(m[3])} if m[3] else set(range(int(m[1]), int(m[2]) + 1))

    kernels = scores = 0
    for body in re.findall(r"^_ZN2rk23gather_attn_wide_kernel\w+:(.*?)^\.Lfunc_end", out.read_text(), re.S | re.M):
        kernels += 1
        written = []                                  # (registers a vector instruction wrote, wait states since)
        for block in re.split(r"^\.LBB\w+:", body, flags=re.M):
            lines = [ln.split(";")[0].split() for ln in block.splitlines()]
            lines = [ln for ln in lines if ln and not ln[0].startswith(".") and not ln[0].endswith(":")]
            ops = [ln[0] for ln in lines]
            if "v_mfma_f32_32x32x16_bf16" in ops and any(op.startswith("ds_read") for op in ops):
                assert not any(op.startswith("scratch_") for op in ops)
            for ln in lines:
                args = [a for a in re.split(r",\s*", " ".join(ln[1:])) if a]
                if ln[0] == "v_mfma_f32_32x32x16_bf16":
                    scores += args[0].startswith("v")
                    used = registers(args[1]) | registers(args[2])
                    assert not any(used & w for w, since in written if since < 2), " ".join(ln)
                states = int(ln[1]) + 1 if ln[0] == "s_nop" else 1
                written = [(w, since + states) for w, since in written if since + states < 2]
                if ln[0].startswith("v_") and not ln[0].startswith("v_mfma") and args:
                    written.append((registers(args[0]), 0))
    assert kernels == 3 and scores == 3 * 32, (kernels, scores)


@pytest.mark.skipif(shutil.which(build.hipcc()) is None, reason="hipcc not found")
@pytest.mark.parametrize("src,with_products", [("block_index.hip", 4), ("index_score.hip", 8), ("mla_attend.hip", 36),
                                               ("gather_attn.hip", 11)])
def test_no_result_of_a_matrix_instruction_is_read_before_it_is_there(src, with_products):
    """On no way through a kernel does an instruction, inline assembly included, come sooner after the matrix instruction whose
    result it reads than the compiler would let it."""
    seen = 0
    for name, body in wait_states.kernels(_compiled(src)[1]):
        products, early = wait_states.early_uses(body)
        seen += products > 0
        assert not early, (name, early[:8])
    assert seen == with_products


def test_reads_of_matrix_results_that_come_too_soon_are_found():
    """wait_states.early_uses on listings with and without the mistake: straight on, around a loop, over a branch, by assembly, of an
    accumulation register, and a write over the result."""
    product = "\tv_mfma_f32_32x32x16_bf16 v[2:17], v[20:23], v[24:27], 0\n"
    use = "\t;;#ASMSTART\n\tv_cvt_pk_bf16_f32 v1, 0, v17 clamp\n\t;;#ASMEND\n"
    other = "\tv_mov_b32_e32 v40, 0\n"
    early = lambda text: [short for _, short in wait_states.early_uses(text + "\ts_endpgm\n")[1]]
    assert early(product + use) == [12] and early(product + "\ts_nop 10\n" + use) == [1] and not early(product + "\ts_nop 11\n" + use)
    assert not early(product + 12 * other + use) and early(product + 11 * other + use) == [1] and early(product + product + use) == [12]
    assert early(use + product) == []
    loop = "\ts_nop 15\n.LBB0_1:\n" + use + "%s\ts_cbranch_scc1 .LBB0_1\n"
    assert early(loop % (product + 9 * other)) == [2] and not early(loop % (product + 11 * other))
    over = product + "\ts_cbranch_scc1 .LBB0_2\n\ts_nop 15\n.LBB0_2:\n" + use
    assert early(over) == [11]
    assert early(product.replace("v[2:17]", "a[2:17]") + "\tv_accvgpr_read_b32 v1, a3\n") == [12]
    assert early(product + "\tv_mov_b32_e32 v9, 0\n") == [12] and not early(product + "\tv_mov_b32_e32 v18, v1\n")
    scaled = "\tv_mfma_scale_f32_32x32x64_f8f6f4 v[2:17], v[20:27], v[30:37], 0, v38, v39 op_sel_hi:[0,0,0]"
    assert early(scaled + "\n" + use) == [20] and early(scaled + " cbsz:4 blgp:4\n" + use) == [12]


@pytest.mark.skipif(shutil.which(build.hipcc()) is None, reason="hipcc not found")
def test_the_code_scorers_sums_run_beside_its_conversions():
    """Of 64 heads two tiles' clamped conversions have, between any two of them, the weight, the rounding and the addition of heads before:
    none of these is put off to the store's branch."""
    body, = [body for name, body in wait_states.kernels(_compiled("block_index.hip")[1]) if "score_blocks_codes_kernel" in name]
    steps, ops = [], None
    for instructions, _ in wait_states.blocks_of(body):
        for op, _, line, _ in instructions:
            if line.endswith(" clamp"):
                steps += [ops] if ops is not None else []
                ops = []
            elif ops is not None:
                ops.append(op)
    steps = [ops for ops in steps if len(ops) < 60]  # (the store between the tiles, and the way around, are longer)
    assert len(steps) >= 118
    late = [ops for ops in steps[3:] if not {"v_mul_f32_e32", "v_cvt_pk_bf16_f32", "v_add_f32_e32"} <= set(ops)]
    assert len(late) <= 3, late[:4]
