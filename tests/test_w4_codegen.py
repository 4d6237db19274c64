"""The 4-wavefront kernel keeps its accumulators in the accumulation registers a0..a255, which it names only
inside inline assembly: the compiler is told they are taken, but nothing stops it from parking other values
there when it runs short of ordinary registers (it did once, in the fused-LayerNorm form, and the accumulators
came out overwritten).  This test compiles the kernels to assembly and checks that the compiler itself never
writes an accumulation register and never spills a vector register.  Scalar registers parked in the lanes of a
vector register (v_writelane / v_readlane) are harmless where they happen once per output tile -- the form of the
fused LayerNorm that walks its tiles keeps two operand streams, the next tile's descriptors and the epilogue's
arguments alive at once -- but not in the steady K loop: no block that holds a whole K tile's 128 MFMAs may contain
one."""
import os
import re
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "general-nvgpu-testing_amd", "csrc")
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")


import pytest


@pytest.fixture(scope="module", params=["gemm_inst_w4.hip", "gemm_inst_w4_kmajor.hip"])
def listing(request, tmp_path_factory):
    """(source, its assembly)"""
    out = tmp_path_factory.mktemp("w4") / "w4.s"
    subprocess.run([HIPCC, "--offload-arch=gfx950", "-O3", "-std=c++17", "-Wno-unused-command-line-argument",
                    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops", "-S", "--cuda-device-only",
                    "-o", str(out), os.path.join(CSRC, request.param)], check=True, capture_output=True, timeout=600)
    return request.param, out.read_text()


# fp16 and bf16, each with three kinds of store, and with two kinds the fused LayerNorm; B as [K][N]: three kinds
KERNELS = {"gemm_inst_w4.hip": 10, "gemm_inst_w4_kmajor.hip": 6}


def test_compiler_never_touches_the_accumulators(listing):
    source, text = listing
    kernels = re.findall(r"^(_ZN4beam16gemmrc_w4_kernel\w+):", text, flags=re.M)
    assert len(kernels) == KERNELS[source], kernels
    assert "v_mfma_f32_16x16x32" in text
    for bad in ("v_accvgpr_write", "v_accvgpr_mov", "scratch_load", "scratch_store"):
        assert bad not in text, f"the compiler emitted {bad} in a 4-wavefront kernel"
    assert set(re.findall(r"\.vgpr_spill_count:\s*(\d+)", text)) == {"0"}
    assert set(re.findall(r"\.private_segment_fixed_size:\s*(\d+)", text)) == {"0"}
    # basic blocks (label to label): the steady K loop is the one with a whole K tile's MFMAs
    steady = [b for b in re.split(r"^\.LBB\d+_\d+:", text, flags=re.M) if b.count("v_mfma_f32_16x16x32") >= 128]
    assert len(steady) >= len(kernels), (len(steady), len(kernels))
    for b in steady:
        assert "v_readlane" not in b and "v_writelane" not in b, "a scalar register is reloaded inside the steady K loop"
    # An inline-assembly statement that writes the scalar condition bit says so: between the statement that sets
    # M0 by an add and the next instruction that tests the bit, something the compiler emitted must have set it.
    lines = [l.strip() for l in text.splitlines()]
    reads = re.compile(r"^(s_cselect_|s_cbranch_scc|s_addc_|s_subb_)")
    writes = re.compile(r"^s_(cmp|cmpk|add|sub|and|or|xor|andn2|orn2|not|lshl|lshr|ashr|bfe|min|max|mul_i32\b.*scc|abs|bitcmp|addk|cmov)")
    adds = [i for i, l in enumerate(lines) if l.startswith("s_add_u32 m0")]
    assert len(adds) > 100
    for i in adds:
        for l in lines[i + 1:]:
            if l.startswith(("s_add_u32 m0", ".LBB", "s_branch", "s_endpgm")) or writes.match(l):
                break
            assert not reads.match(l), f"line {i}: `{l}` tests the condition bit an M0 add in inline assembly has overwritten"


def scalars(text):
    regs = {int(r) for r in re.findall(r"\bs(\d+)\b", text)}
    for first, last in re.findall(r"\bs\[(\d+):(\d+)\]", text):
        regs |= set(range(int(first), int(last) + 1))
    if re.search(r"\bvcc\b", text):
        regs.add("vcc")
    return regs


def too_early(lines):
    """Memory instructions of `lines` that read a scalar register less than 5 wait states after a vector instruction wrote it
    (v_readlane, which restores a parked one, v_readfirstlane, a compare into a scalar pair), and how many restores there are.
    Taken branches start with what the lines in front of the branch left, which its label finds written too."""
    at, written, restores, bad = 0, {}, 0, []
    behind = {}  # label: registers written in front of a branch to it, and how long before
    for line in lines:
        line = line.split(";")[0].strip()
        if line.endswith(":"):
            for r, age in behind.pop(line[:-1], {}).items():
                written[r] = max(written.get(r, -100), at - age)
        if not line or line.startswith(".") or line.endswith(":"):
            continue
        op, _, args = line.replace("\t", " ").partition(" ")
        first, _, rest = args.partition(",")
        at += int(args, 0) + 1 if op == "s_nop" else 1
        if op.startswith(("buffer_", "global_")):
            late = [r for r in scalars(args) if r in written and at - written[r] - 1 < 5]
            if late:
                bad.append(f"`{line}` reads s{late} {at - written[late[0]] - 1} wait states after a vector instruction wrote it")
        elif op.startswith("v_"):
            if op in ("v_readlane_b32", "v_readfirstlane_b32"):
                restores += 1
            written.update((r, at) for r in scalars(first))
            if op.startswith("v_cmp") and "_e32" in op:
                written["vcc"] = at
        elif op.startswith(("s_branch", "s_cbranch")):
            ages = behind.setdefault(args.strip(), {})
            for r, when in written.items():
                if at - when <= 5:
                    ages[r] = min(ages.get(r, 100), at - when)
        elif op.startswith("s_") and not op.startswith(("s_cmp", "s_bitcmp", "s_nop", "s_waitcnt", "s_barrier", "s_setprio")):
            for r in scalars(first):
                written.pop(r, None)
    return bad, restores


def test_restored_scalars_reach_memory_instructions_late_enough(listing):
    """A memory instruction may read a scalar register that a vector instruction wrote only 5 wait states later.  The compiler
    sees to that for its own instructions and does not look into inline assembly: an order of the kernels' arguments that made it
    park more scalars put a restored one right in front of a load there, and the fused LayerNorm came out wrong (256 x 512 x
    256).  The source keeps the distance for a stream's first load behind a boundary of output tiles; this looks at every load."""
    source, text = listing
    lines = text.splitlines()
    bad, restores = too_early(lines)
    # back edges: once more around every loop, from the branch to the label and on
    labels = {l.split(":")[0]: i for i, l in enumerate(lines) if re.match(r"^\.LBB\d+_\d+:", l)}
    for i, l in enumerate(lines):
        branch = re.match(r"^\s*s_c?branch\w*\s+(\.LBB\d+_\d+)", l)
        if branch and labels.get(branch[1], i) < i:
            bad += too_early(lines[max(0, i - 12):i] + lines[labels[branch[1]] + 1:labels[branch[1]] + 13])[0]
    assert not bad, bad[:4]
    assert restores > 50
    fresh = re.findall(r"s_nop 4\n\s*buffer_load_dwordx4 [^\n]* lds", text)
    assert len(fresh) >= 5 * KERNELS[source], (len(fresh), source)


@pytest.mark.parametrize("lines,finds", [
    (["v_readlane_b32 s5, v1, 0", "s_nop 3", "buffer_load_dwordx4 v0, s[4:7], 0 offen lds"], 1),
    (["v_readlane_b32 s5, v1, 0", "s_nop 4", "buffer_load_dwordx4 v0, s[4:7], 0 offen lds"], 0),
    (["v_readlane_b32 s5, v1, 0", "s_cmp_eq_u32 s5, 0", "buffer_load_dwordx4 v0, s[4:7], 0 offen lds"], 1),
    (["v_readlane_b32 s5, v1, 0", "s_mov_b32 s5, s9", "buffer_load_dwordx4 v0, s[4:7], 0 offen lds"], 0),
    (["v_cmp_gt_i32_e64 s[8:9], v1, v2", "buffer_load_dwordx4 v0, s[4:7], s8 offen lds"], 1),
    (["v_readlane_b32 s5, v1, 0", "s_cbranch_scc1 .LBB0_2", "s_mov_b32 s5, 0", ".LBB0_2:", "buffer_load_dwordx4 v0, s[4:7], 0 offen lds"], 1),
])
def test_the_scan_finds_what_it_looks_for(lines, finds):
    assert len(too_early(lines)[0]) == finds
