"""Properties of the compiled gfx950 code that the source relies on but the compiler does not guarantee (CPU only: hipcc
cross-compiles without a GPU).

attn_exact.hip issues v_fmac_f64 with a DPP operand from inline assembly.  The compiler's hazard recognizer does not look
into asm blocks, so the idle cycles a DPP read needs are written by hand (two, in front of every group, against a vector
write of the DPP source) or avoided by construction (five behind a vector instruction that writes EXEC: the kernel must
not contain one)."""
import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "bunker_amd", "csrc")
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")


def _makefile_flags(source):
    """The flags that the Makefile compiles ``source`` with: HIPFLAGS and, where its object has them, EXTRA."""
    mk = open(os.path.join(CSRC, "Makefile")).read()
    flags = re.search(r"^HIPFLAGS \?= (.*?)(?<!\\)$", mk, flags=re.M | re.S).group(1).replace("\\\n", " ").replace("$(ARCH)", "gfx950").split()
    for targets, extra in re.findall(r"^(build/[^:=%$]*): EXTRA := (.*)$", mk, flags=re.M):
        if "build/" + source.replace(".hip", ".o") in targets.split():
            flags += extra.split()
    return flags


def _compile_to_asm(tmp_path_factory, source):
    if not (os.path.exists(HIPCC) or shutil.which(HIPCC)):
        pytest.skip("hipcc not found")
    out = str(tmp_path_factory.mktemp("isa") / (source + ".s"))
    subprocess.check_call([HIPCC, *_makefile_flags(source), "-S", "--cuda-device-only", "-o", out, os.path.join(CSRC, source)],
                          stderr=subprocess.DEVNULL)
    return open(out).read()


def test_the_checks_compile_what_the_makefile_compiles():
    """Every source with the command line that make would run for it (a source checked without its own flags is other code)."""
    out = subprocess.run(["make", "-C", CSRC, "-n", "-B"], check=True, capture_output=True, text=True).stdout
    lines = {m.group(2): m.group(1).split() for m in re.finditer(r"hipcc (.*) -c (\S+\.hip) -o", out.replace("\\\n", " "))}
    assert len(lines) >= 16 and any("-mllvm" in f for f in lines.values())
    for source, flags in lines.items():
        assert _makefile_flags(source) == flags, source


@pytest.fixture(scope="module")
def exact_asm(tmp_path_factory):
    return _compile_to_asm(tmp_path_factory, "attn_exact.hip")


def _kernels(asm):
    """name -> body of every kernel of the file"""
    out = {}
    for m in re.finditer(r"^(_ZN2bk\w+):[^\n]*\n(.*?)^\.Lfunc_end", asm, flags=re.M | re.S):
        out[m.group(1)] = m.group(2)
    return out


def test_dpp_groups_in_the_exact_attention_are_hazard_free(exact_asm):
    ks = {k: v for k, v in _kernels(exact_asm).items() if "attn_exact_kernel" in k}
    assert len(ks) == 4                                         # plain / nontemporal loads x with / without the folded preparation
    for name, body in ks.items():
        n_dpp = len(re.findall(r"\bv_fmac_f64_dpp\b", body))
        assert n_dpp >= 512 and n_dpp % 8 == 0, (name, n_dpp)
        # no vector instruction writes EXEC anywhere in the kernel
        assert not re.search(r"\bv_cmpx", body), name
        # every DPP instruction sits in an asm block that opens with the two idle cycles, eight to a block
        blocks = re.findall(r";;#ASMSTART\n(.*?);;#ASMEND", body, flags=re.S)
        dpp_blocks = [b for b in blocks if "v_fmac_f64_dpp" in b]
        assert sum(len(re.findall(r"v_fmac_f64_dpp", b)) for b in dpp_blocks) == n_dpp
        for b in dpp_blocks:
            lines = [l.strip() for l in b.strip().splitlines()]
            assert lines[0] == "s_nop 1" and len(lines) == 9 and all(l.startswith("v_fmac_f64_dpp") for l in lines[1:]), b
            # the broadcast source is read, never written, inside the block
            src = {re.match(r"v_fmac_f64_dpp (v\[\d+:\d+\]), (v\[\d+:\d+\]),", l).group(2) for l in lines[1:]}
            dst = {re.match(r"v_fmac_f64_dpp (v\[\d+:\d+\]),", l).group(1) for l in lines[1:]}
            assert len(src) == 1 and not (src & dst), b
        # no register spills: the kernel is sized for 128 registers per lane and 4 waves per SIMD
        meta = re.search(r"\.name:\s+%s\n(.*?)\.wavefront_size" % re.escape(name), exact_asm, flags=re.S).group(1)
        assert int(re.search(r"\.vgpr_count:\s+(\d+)", meta).group(1)) <= 128
        assert int(re.search(r"\.vgpr_spill_count:\s+(\d+)", meta).group(1)) == 0


@pytest.mark.parametrize("source,kernels,transfer,mfma,min_mfma", [
    ("attn_prefill.hip", ["attn_prefill_kernel"], "global_load_lds_dwordx4", "v_mfma_f32_32x32x16_bf16", 64),
    ("gdn_chunk.hip", ["gdn_chunk_wu_kernel", "gdn_chunk_state_kernel", "gdn_chunk_out_kernel"], "global_load_lds_dword", "v_mfma_f32_32x32x2_f32", 32),
])
def test_lds_transfers_written_as_instructions_own_m0(tmp_path_factory, source, kernels, transfer, mfma, min_mfma):
    """lds_dma16 / lds_dma4 (common.h) set m0 themselves and tell the compiler so, but m0 is a register the compiler
    reserves: the kernels that use them must contain no other use of it, every write of m0 must be followed (one idle
    cycle later) by the transfer that reads it, and the compiler's own form of the transfer — behind which it waits for
    the whole transfer before the next LDS access — must not have come back.  Also: no vector spills, no scalar spills
    in the blocks that issue matrix instructions, no scratch, and the matrix instruction the kernel is built around is
    there."""
    asm = _compile_to_asm(tmp_path_factory, source)
    bodies = _kernels(asm)
    for kname in kernels:
        name, body = next((k, v) for k, v in bodies.items() if kname in k)
        lines = [l.strip() for l in body.split("\n") if l.strip() and not l.strip().startswith((";", "."))]
        m0 = [i for i, l in enumerate(lines) if re.search(r"\bm0\b", l)]
        assert m0, name
        for i in m0:
            assert lines[i].startswith("s_mov_b32 m0,"), (name, lines[i])
            assert lines[i + 1].startswith("s_nop") and lines[i + 2].startswith(transfer + " "), (name, lines[i:i + 3])
        assert sum(l.startswith(transfer + " ") for l in lines) == len(m0), name
        assert sum(l.startswith(mfma + " ") for l in lines) >= min_mfma, name
        meta = re.search(r"\.name:\s+%s\n(.*?)\.wavefront_size" % re.escape(name), asm, flags=re.S).group(1)
        assert int(re.search(r"\.vgpr_spill_count:\s+(\d+)", meta).group(1)) == 0, name
        # scalar registers: a handful of spills in the set-up code are tolerated, none where matrix instructions are issued
        # (a spilled scalar is a lane read or write in the wave's instruction stream)
        assert int(re.search(r"\.sgpr_spill_count:\s+(\d+)", meta).group(1)) <= 8, name
        for block in re.split(r"^\.LBB\d+_\d+:", body, flags=re.M):
            if block.count(mfma + " ") >= 4:
                assert "v_readlane_b32" not in block and "v_writelane_b32" not in block, name
        assert int(re.search(r"\.private_segment_fixed_size:\s+(\d+)", meta).group(1)) == 0, name


@pytest.mark.parametrize("source,kernel,kernarg_sizes", [
    # SwiGLU pair 52 (padded to 56), one matrix 64, several matrices 104 / 128 with the convolution's operands, general
    # 176 / 208; no implicit arguments behind them (the kernel reads the grid size from its block, not from gridDim)
    ("gemv_fused.hip", "gemv_fused_kernel", {56, 64, 104, 128, 176, 208}),
    ("gdn.hip", "gdn_slab_kernel", {80}),
    ("gemm_mfma.hip", "gemm_q4k_q8_1_mfma_kernel", {56, 64, 184}),
])
def test_argument_blocks_stay_compact_and_in_registers(tmp_path_factory, source, kernel, kernarg_sizes):
    """The decode step's kernels take the smallest by-value argument block their form needs (a launch pays for every
    64-byte line of it) and rebuild the general block in registers.  That only works while the compiler keeps the rebuilt
    block out of private memory and LDS: no kernel of these families may have a private segment, and every argument-block
    size the launchers rely on must be there."""
    asm = _compile_to_asm(tmp_path_factory, source)
    seen = set()
    for m in re.finditer(r"\.kernarg_segment_size:\s+(\d+)\n(.*?)\.name:\s+(\S+)\n(.*?)\.wavefront_size", asm, flags=re.S):
        if kernel not in m.group(3):
            continue
        meta = m.group(2) + m.group(4)
        seen.add(int(m.group(1)))
        assert int(re.search(r"\.private_segment_fixed_size:\s+(\d+)", meta).group(1)) == 0, m.group(3)
        assert int(re.search(r"\.vgpr_spill_count:\s+(\d+)", meta).group(1)) == 0, m.group(3)
    assert seen and seen <= kernarg_sizes and min(seen) == min(kernarg_sizes), seen


def test_range_checked_loads_carry_their_whole_offset_in_the_lane_operand(tmp_path_factory):
    """gemv_rows.hip lets the range check of a buffer resource answer for the pieces past the end of the weight and activation rows.
    That check is defined over the lane's offset and the immediate one; a scalar offset operand is not part of it, so it has to be 0."""
    asm = _compile_to_asm(tmp_path_factory, "gemv_rows.hip")
    bodies = {k: v for k, v in _kernels(asm).items() if "gemv_rows" in k}
    assert len(bodies) >= 13
    for name, body in bodies.items():
        loads = re.findall(r"^\s*buffer_load_\w+ (.*)$", body, flags=re.M)
        assert loads, name
        for l in loads:
            assert re.match(r"v\[\d+:\d+\], v\d+, s\[\d+:\d+\], 0 offen\b", l), (name, l)


def test_prompt_attention_in_double_precision_walks_its_pages_without_scratch(tmp_path_factory):
    """attn_prefill_exact.hip is sized for 256 registers and two workgroups a CU.  The forms of 2, 4 and 8 heads use no scratch; that of one
    head parks a single constant, outside the page loop (the blocks with matrix instructions, and what lies between them)."""
    asm = _compile_to_asm(tmp_path_factory, "attn_prefill_exact.hip")
    bodies = {k: v for k, v in _kernels(asm).items() if "attn_prefill_exact_kernel" in k}
    assert len(bodies) == 4
    for name, body in bodies.items():
        meta = re.search(r"\.name:\s+%s\n(.*?)\.wavefront_size" % re.escape(name), asm, flags=re.S).group(1)
        spills = int(re.search(r"\.vgpr_spill_count:\s+(\d+)", meta).group(1))
        assert spills <= (2 if "ILi1E" in name else 0), (name, spills)
        assert int(re.search(r"\.sgpr_spill_count:\s+(\d+)", meta).group(1)) == 0, name
        first, last = body.index("v_mfma_f64_16x16x4"), body.rindex("v_mfma_f64_16x16x4")
        assert "scratch_" not in body[first:last], name


def _registers(operand):
    m = re.match(r"v\[(\d+):(\d+)\]$|v(\d+)$", operand)
    return set() if not m else set(range(int(m.group(1)), int(m.group(2)) + 1)) if m.group(1) else {int(m.group(3))}


def test_nothing_is_placed_in_the_results_of_a_matrix_instruction_in_flight(tmp_path_factory):
    """gemm_mfma.hip adds up in asm blocks between a matrix instruction and the first read of its results.  The compiler keeps the distance
    that the matrix unit needs before a register of its results may be written again, but not from what it cannot look into:
    up to the last of these blocks no instruction may write any of the sixteen registers (also those that a narrow tile ignores)."""
    asm = _compile_to_asm(tmp_path_factory, "gemm_mfma.hip")
    bodies = {k: v for k, v in _kernels(asm).items() if "gemm_q4k_q8_1_mfma_kernel" in k}
    assert len(bodies) >= 15
    for name, body in bodies.items():
        ins = [l.strip().replace(",", "").split() for l in body.split("\n") if re.match(r"\s+[a-z]\w+(\s|$)", l)]
        checked = 0
        for i, first in enumerate(ins):
            if not first[0].startswith("v_mfma_i32_32x32x32_i8"):
                continue
            results, written = _registers(first[1]), None
            assert len(results) == 16
            for x in ins[i + 1:]:
                if x[0].startswith(("s_cbranch", "s_branch", "s_endpgm")):
                    break
                writes = len(x) > 1 and not x[0].startswith(("ds_write", "global_store", "s_"))
                if any(_registers(r) & results for r in x[2 if writes else 1:]):
                    break
                if writes and _registers(x[1]) & results:
                    written = written or x
                    results = results - _registers(x[1])
                if x[0] == "v_mad_i64_i32":
                    assert not written, (name, first, written)
                    checked += 1
        assert checked >= 7 * 4, (name, checked)


def test_results_of_the_tiles_matmul_are_first_read_where_the_compiler_sees_it(tmp_path_factory):
    """gemm_tiles.hip multiplies and adds in asm blocks.  The compiler keeps the distance that the results of a matrix instruction need
    before they are read or written, but does not look into the blocks: of every int8 product some result must be read by
    an instruction outside them first, and none may be written before that.  Three waves share a SIMD: 168 registers, no scratch."""
    asm = _compile_to_asm(tmp_path_factory, "gemm_tiles.hip")
    bodies = {k: v for k, v in _kernels(asm).items() if "gemm_q4k_q8_1_tiles_kernel" in k}
    assert len(bodies) == 2
    for name, body in bodies.items():
        meta = re.search(r"\.name:\s+%s\n(.*?)\.wavefront_size" % re.escape(name), asm, flags=re.S).group(1)
        assert int(re.search(r"\.vgpr_count:\s+(\d+)", meta).group(1)) <= 168, name
        assert int(re.search(r"\.vgpr_spill_count:\s+(\d+)", meta).group(1)) == 0, name
        assert int(re.search(r"\.private_segment_fixed_size:\s+(\d+)", meta).group(1)) == 0, name
        ins, inside = [], False
        for l in body.split("\n"):
            inside = True if "#ASMSTART" in l else False if "#ASMEND" in l else inside
            if re.match(r"\s+[a-z]\w+(\s|$)", l):
                ins.append((inside, l.strip().replace(",", "").split()))
        checked = 0
        for i, (_, first) in enumerate(ins):
            if not first[0].startswith("v_mfma_i32_16x16x32_i8"):
                continue
            results = _registers(first[1])
            assert len(results) == 4
            for in_block, x in ins[i + 1:]:
                if x[0].startswith(("s_cbranch", "s_branch", "s_endpgm")):
                    break
                writes = len(x) > 1 and not x[0].startswith(("ds_write", "global_store", "s_"))
                if any(_registers(r) & results for r in x[2 if writes else 1:]):
                    assert not in_block, (name, first, x)
                    checked += 1
                    break
                assert not (writes and _registers(x[1]) & results), (name, first, x)
        assert checked >= 2 * 32, (name, checked)


def test_the_numbered_rows_gemv_fits_the_registers_of_its_waves(tmp_path_factory):
    """gemv.hip: every form of the flat kernel and of the f32 kernel without scratch.  A spilled piece of the next step's weights is waited for before
    the step at hand is folded."""
    asm = _compile_to_asm(tmp_path_factory, "gemv.hip")
    names = [n for n in _kernels(asm) if "gemv_q4k_q8_1_flat_kernel" in n or "gemv_q4k_f32_lds_kernel" in n]
    assert len(names) == 9 * 3 + 4
    for name in names:
        meta = re.search(r"\.name:\s+%s\n(.*?)\.wavefront_size" % re.escape(name), asm, flags=re.S).group(1)
        assert int(re.search(r"\.vgpr_spill_count:\s+(\d+)", meta).group(1)) == 0, name
        assert int(re.search(r"\.private_segment_fixed_size:\s+(\d+)", meta).group(1)) == 0, name
