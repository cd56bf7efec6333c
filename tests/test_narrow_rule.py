"""The rule that sends products with a narrow side to their kernel (csrc/narrow_rule.hpp), compiled
for the host: what it takes fits a launch, and every K-step belongs to exactly one part."""
import ctypes
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "cumpsgemm_amd", "csrc")
CUS = 256


@pytest.fixture(scope="module")
def plan(tmp_path_factory):
    d = tmp_path_factory.mktemp("rule")
    (d / "rule.cpp").write_text("""
        #include "narrow_rule.hpp"
        extern "C" void plan(int bf16x3, uint32_t wide, uint32_t few, uint32_t k, uint32_t cus, uint32_t *out) {
          const cumpsgemm_amd::NarrowPlan p = cumpsgemm_amd::plan_narrow(bf16x3 != 0, wide, few, k, cus);
          out[0] = p.waves, out[1] = p.chunks, out[2] = p.steps_per_chunk;
        }""")
    so = d / "rule.so"
    subprocess.check_call(["g++", "-std=c++17", "-shared", "-fPIC", "-I", CSRC, "-o", str(so), str(d / "rule.cpp")])
    lib = ctypes.CDLL(str(so))

    def call(bf16x3, wide, few, k):
        """(waves, parts of K, K-steps of a part), or None: the tiled kernels."""
        out = (ctypes.c_uint32 * 3)()
        lib.plan(int(bf16x3), wide, few, k, CUS, out)
        return tuple(out) if out[1] else None
    return call


@pytest.mark.parametrize("bf16x3", [False, True])
def test_a_launch_holds_what_the_rule_takes(plan, bf16x3):
    taken = 0
    for wide in (1024, 1025, 8192, 8193, 16352, 16353, 1 << 20, (1 << 28) - 64, (1 << 28) - 31, 1 << 28, 1 << 30, (1 << 31) - 1):
        for few in (1, 16, 17, 32):
            for k in (1, 31, 32, 33, 1000, 1024, 8192, 131072, (1 << 31) - 1):
                p = plan(bf16x3, wide, few, k)
                if p is None:
                    continue
                taken += 1
                waves, chunks, steps = p
                # HIP refuses 2^32 threads or more along an axis
                assert (wide + 31) // 32 * waves * 64 < 1 << 32, (wide, few, k)
                assert waves in (8, 16) and chunks <= 65535
                assert steps * chunks >= k // 32 and steps * (chunks - 1) < max(1, k // 32), (wide, few, k)
    assert taken > 20
