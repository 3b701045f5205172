"""What the grouped GEMMs rely on in the code generated for them, read from
the assembly of gemm_kernels.hip compiled here (no GPU needed)."""
import os
import re
import subprocess

import pytest

from flash_deepseek_amd import build as B

# the project's own schedule, and another of the compiler's schedulers: what
# only the source may promise must hold under both
SCHEDULERS = {"default": [], "max-ilp": ["-mllvm", "-amdgpu-sched-strategy=max-ilp"]}


@pytest.fixture(scope="module", params=list(SCHEDULERS))
def assembly(request, tmp_path_factory):
    """{kernel: its assembly lines}"""
    try:
        hipcc = B._hipcc()
    except RuntimeError as e:
        pytest.skip(str(e))
    out = str(tmp_path_factory.mktemp("gemm") / "gemm.s")
    subprocess.run([hipcc, *B.CXXFLAGS, *SCHEDULERS[request.param], "--cuda-device-only", "-S",
                    os.path.join(B.CSRC, "gemm_kernels.hip"), "-o", out], check=True, capture_output=True)
    kernels, lines = {}, None
    with open(out) as f:
        for ln in f:
            if re.match(r"_ZN\w+:", ln):
                lines = kernels.setdefault(ln.split(":")[0], [])
            elif lines is not None:
                lines.append(ln.strip())
    gemms = {k: v for k, v in kernels.items() if "k_qgemm" in k}
    assert len(gemms) == 5
    return gemms


def test_counted_waits_cover_the_direct_loads(assembly):
    """A wait that leaves the N youngest loads in flight stands for "the token
    operands have landed in LDS": none of the last N loads before it may be a
    direct global -> LDS load."""
    waits = 0
    for kernel, lines in assembly.items():
        loads, in_asm = [], False
        for ln in lines:
            in_asm = (in_asm or "#ASMSTART" in ln) and "#ASMEND" not in ln
            if re.match(r"(buffer|global|scratch|flat)_(load|store|atomic)", ln):
                loads.append(ln)
            m = re.match(r"s_waitcnt vmcnt\((\d+)\)$", ln)
            if m and in_asm and int(m[1]):
                waits += 1
                assert not any(re.search(r"\blds\b", x) for x in loads[-int(m[1]):]), (kernel, ln, loads[-int(m[1]):])
    assert waits >= 5 * 3


def test_plane_sums_read_after_a_fence(assembly):
    """The packed bodies add a token's three planes across lanes through LDS:
    between a tile's LDS writes and the reads of other lanes' values, and again
    before the next tile's writes, stands a wave barrier (with its fences)."""
    epilogues = 0
    for kernel, lines in assembly.items():
        if "ILi3E" not in kernel:  # three planes
            continue
        ops = ""
        for ln in lines:
            ops += ("b" if "wave barrier" in ln else "w" if ln.startswith("ds_write") else
                    "r" if ln.startswith("ds_read") else "S" if re.match(r"(global|buffer)_store", ln) else "")
        tiles = re.findall(r"w(b*)r+S(b*)", ops)  # a tile's values, the sums over them, the output
        tiles = [t for t in tiles if t[1]]  # the other bodies store what they hold
        epilogues += len(tiles)
        assert tiles and all(t == ("b", "b") for t in tiles), (kernel, ops)
    assert epilogues >= 3 * 4


def test_nothing_spills(assembly):
    """No GEMM keeps registers in scratch memory: a reload inside the
    contraction waits for every older load and so drains the weight stream."""
    for kernel, lines in assembly.items():
        touched = [ln for ln in lines if ln.startswith("scratch_")]
        assert not touched, (kernel, len(touched), touched[:3])
