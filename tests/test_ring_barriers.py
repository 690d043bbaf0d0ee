"""The LDS rings of the copy pipelines: at every barrier of their kernels the wave has waited for its own LDS reads
(lgkmcnt(0)), as past the barrier another wave's copy may overwrite the stage they come from. Checked in the gfx950
assembly of the sources as built, so that it does not rest on where the compiler places the products."""

import concurrent.futures as cf
import re
import subprocess

import pytest

from vesper_amd.build import CSRC, HIP_FLAGS, hipcc

# source, kernel, least number of barriers
RINGS = [("mx_moe", "gateup_kernel", 6), ("mx_prefill", "gateup_exact_kernel", 8), ("mx_prefill", "grouped_down_kernel", 4),
         ("mx_fp8", "fp8_gemm_kernel", 8)]


@pytest.fixture(scope="module")
def assembly(tmp_path_factory):
    out = tmp_path_factory.mktemp("asm")

    def compile_one(name):
        path = out / f"{name}.s"
        subprocess.run([hipcc(), *HIP_FLAGS, "--cuda-device-only", "-S", str(CSRC / f"{name}.hip"), "-o", str(path)],
                       check=True, stdout=subprocess.DEVNULL, stderr=subprocess.DEVNULL)
        return name, path.read_text()

    with cf.ThreadPoolExecutor() as pool:
        return dict(pool.map(compile_one, sorted({source for source, _, _ in RINGS})))


def barriers(text, kernel):
    """For each barrier of the kernel's instances, the instructions of its basic block before it, nearest first."""
    inside, block, found = False, [], []
    for line in text.splitlines():
        line = line.split(";")[0].strip()
        label = re.match(r"^(\S+):$", line)
        if label:
            if label.group(1).startswith("_Z"):
                inside = kernel in label.group(1)
            block = []
        elif inside and line and not line.startswith("."):
            if line.startswith("s_barrier"):
                found.append(block[::-1])
                block = []
            elif line.startswith(("s_cbranch", "s_branch")):
                block = []
            else:
                block.append(line)
    return found


@pytest.mark.parametrize("source,kernel,least", RINGS)
def test_lds_reads_are_waited_for_at_every_barrier(assembly, source, kernel, least):
    found = barriers(assembly[source], kernel)
    assert len(found) >= least
    for block in found:
        waited = False
        for line in block:
            if line.startswith("s_waitcnt") and "lgkmcnt(0)" in line:
                waited = True
                break
            if line.startswith("ds_"):
                break
        assert waited, f"{kernel}: a barrier with no wait for the LDS reads before it: {block[:4]}"
