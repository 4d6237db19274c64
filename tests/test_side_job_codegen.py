"""The K loop that carries the side job keeps its loads in flight: the compiler waits for the job's own (vmcnt of what is younger), and
drains them all (vmcnt(0)) in no K tile.  It did once, in the loop of the 8-byte units of the 256 x 128 tile, for a loop in the epilogue
behind it (1117 x 6352 x 7616 with 58 Mi elements 144 -> 161 us), which no result shows."""
import os
import re
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "general-nvgpu-testing_amd", "csrc")
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
SIDE = 4  # kEpiStoreSide


def inner_loops(body):
    lines = body.splitlines()
    labels = {m[1]: i for i, l in enumerate(lines) if (m := re.match(r"^(\.LBB\d+_\d+):", l))}
    for i, l in enumerate(lines):
        branch = re.match(r"^\s+s_c?branch\w*\s+(\.LBB\d+_\d+)", l)
        if branch and labels.get(branch[1], i) < i:
            loop = "\n".join(lines[labels[branch[1]]:i])
            if loop.count("v_mfma") == 32 and loop.count("s_barrier") == 1:
                yield loop


def test_side_job_loops_never_drain(tmp_path):
    out = tmp_path / "side.s"
    subprocess.run([HIPCC, "--offload-arch=gfx950", "-O3", "-std=c++17", "-Wno-unused-command-line-argument",
                    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops", "-S", "--cuda-device-only",
                    "-o", str(out), os.path.join(CSRC, "gemm_inst_256x128_64x64.hip")], check=True, capture_output=True, timeout=600)
    text = out.read_text()
    kernels = re.findall(rf"^(_ZN4beam13gemmrc_kernelIDF16\w?Li256ELi128ELi4ELi2ELi{SIDE}E\w+):", text, flags=re.M)
    assert len(kernels) == 4, kernels  # two types, two depths
    for k in kernels:
        start = text.index("\n" + k + ":")
        loops = list(inner_loops(text[start:text.index(".Lfunc_end", start)]))
        carrying = [l for l in loops if "v_rcp_f32" in l]
        assert len(carrying) >= 2, (k, len(loops))
        for l in carrying:
            waits = [int(n) for n in re.findall(r"vmcnt\((\d+)\)", l)]
            # (the 16-byte units' loop lies around the tail's, which may drain)
            assert 0 not in waits or len(l.splitlines()) > 500, (k, waits)
