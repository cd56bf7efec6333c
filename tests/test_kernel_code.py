"""What the compiler made of the GEMM kernels, read back from the built library."""
import os
import re
import shutil
import subprocess

import pytest

import cumpsgemm_amd

OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    """Name of each kernel -> its instructions, (mnemonic and operands, address, branch target or None)."""
    if not os.path.exists(OBJDUMP):
        pytest.skip("no llvm-objdump")
    lib = os.path.join(os.path.dirname(cumpsgemm_amd.__file__), "libcumpsgemm.so")
    d = tmp_path_factory.mktemp("code")
    shutil.copy(lib, d)
    subprocess.check_call([OBJDUMP, "--offloading", "libcumpsgemm.so"], cwd=d, stdout=subprocess.DEVNULL)
    out = {}
    for f in sorted(os.listdir(d)):
        if not f.endswith("gfx950"):
            continue
        code = None
        for line in subprocess.run([OBJDUMP, "-d", f], cwd=d, capture_output=True, text=True, check=True).stdout.split("\n"):
            head = re.match(r"^[0-9a-f]+ <(\w+)>:", line)
            if head:
                code = out.setdefault(head.group(1), [])
            elif line.startswith("\t") and code is not None and "//" in line:
                text, note = line.strip().split("//", 1)
                at = int(note.split(":")[0], 16)
                jump = re.match(r"s_cbranch_\w+ (\d+)", text)
                off = int(jump.group(1)) if jump else 0
                code.append((text.strip(), at, at + 4 + 4 * (off - 65536 if off >= 32768 else off) if jump else None))
    return out


def loops_over_lane_values(code):
    """Loads that run once per distinct value of an operand that must be uniform: a few instructions that
    take one lane's value, load for the lanes that share it and branch back while any are left."""
    found = 0
    for i, (text, at, target) in enumerate(code):
        if text.startswith("s_cbranch_execnz") and target <= at:
            body = [t for t, a, _ in code[max(0, i - 40):i] if a >= target]
            found += any(t.startswith("buffer_load") for t in body) and any(t.startswith("v_readfirstlane") for t in body)
    return found


def test_no_load_of_a_gemm_kernel_is_a_loop_over_lane_values(kernels):
    gemm = {n: c for n, c in kernels.items() if "gemm_tcec_kernel" in n or "narrow_kernel" in n}
    assert len(gemm) > 200 and all(any("v_mfma" in t for t, _, _ in c) for c in gemm.values())
    bad = {n: k for n, k in ((n, loops_over_lane_values(c)) for n, c in gemm.items()) if k}
    assert not bad, bad


def scratch_accesses_of_k_loops(code):
    """Scratch loads and stores inside loops that multiply."""
    found = 0
    for i, (text, at, target) in enumerate(code):
        if target is not None and target <= at:
            body = [t for t, a, _ in code[:i] if a >= target]
            if any(t.startswith("v_mfma") for t in body):
                found += sum(t.startswith("scratch_") for t in body)
    return found


def test_scaled_large_kernel_of_k_contiguous_operands_keeps_its_addresses_in_registers(kernels):
    # GemmCfg<FP16TCEC, real, K-contiguous, K-contiguous, 256, 128, 64, 64, 2, DEEP, one tile, SCALED, in-loop>
    (code,) = [c for n, c in kernels.items() if "PrecE0ELb0ELb1ELb1ELi256ELi128ELi64ELi64ELi2ELb1ELb0ELb1ELb0E" in n]
    assert scratch_accesses_of_k_loops(code) == 0


def first_loads_of_k_loops(code):
    """Share of a loop's MFMAs that stand before its first global load, for every loop that multiplies and loads."""
    out = []
    for i, (text, at, target) in enumerate(code):
        if target is not None and target <= at:
            body = [t for t, a, _ in code[:i + 1] if a >= target]
            mfma = [j for j, t in enumerate(body) if t.startswith("v_mfma")]
            loads = [j for j, t in enumerate(body) if t.startswith(("global_load", "buffer_load"))]
            if mfma and loads:
                out.append(sum(j < loads[0] for j in mfma) / len(mfma))
    return out


@pytest.mark.parametrize("tile", ["Lb0ELb1ELb1ELi256ELi128ELi64ELi64E", "Lb0ELb1ELb1ELi128ELi128ELi64ELi32E",
                                  "Lb1ELb1ELb1ELi128ELi64ELi32ELi32E"])
def test_loads_of_two_k_contiguous_bf16x2_operands_are_not_left_behind_the_split(kernels, tile):
    """The one-tile kernels ask for a step's operands while they split the one before it."""
    # GemmCfg<bf16x2, real / complex, K-contiguous, K-contiguous, tile, 2, DEEP, one tile, not scaled, in-loop>
    found = [c for n, c in kernels.items() if "PrecE3E" + tile in n and "Li2ELb1ELb0ELb0ELb0E" in n]
    assert len(found) == 1
    first = first_loads_of_k_loops(found[0])
    assert first and min(first) <= 0.6, first
