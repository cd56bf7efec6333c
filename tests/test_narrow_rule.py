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
        extern "C" void plan(int bf16x3, int big_kc, int small_kc, uint32_t wide, uint32_t few, uint32_t k,
                             uint32_t cus, uint32_t *out) {
          const cumpsgemm_amd::NarrowPlan p =
              cumpsgemm_amd::plan_narrow(bf16x3 != 0, big_kc != 0, small_kc != 0, wide, few, k, cus);
          out[0] = p.waves, out[1] = p.chunks, out[2] = p.steps_per_chunk;
        }""")
    so = d / "rule.so"
    subprocess.check_call(["g++", "-std=c++17", "-shared", "-fPIC", "-I", CSRC, "-o", str(so), str(d / "rule.cpp")])
    lib = ctypes.CDLL(str(so))

    def call(bf16x3, wide, few, k, op="TN"):
        """(waves, parts of K, K-steps of a part), or None: the tiled kernels.  op: as of wide x k times k x few."""
        out = (ctypes.c_uint32 * 3)()
        lib.plan(int(bf16x3), int(op[0] == "T"), int(op[1] == "N"), wide, few, k, CUS, out)
        return tuple(out) if out[1] else None
    return call


@pytest.mark.parametrize("bf16x3", [False, True])
def test_a_launch_holds_what_the_rule_takes(plan, bf16x3):
    taken = 0
    for wide in (1024, 1025, 8192, 8193, 16352, 16353, 1 << 20, (1 << 28) - 64, (1 << 28) - 31, 1 << 28, 1 << 30, (1 << 31) - 1):
        for few in (1, 16, 17, 32):
            for k in (1, 31, 32, 33, 1000, 1024, 8192, 131072, (1 << 31) - 1):
                for op in ("TN", "NN", "TT", "NT"):
                    p = plan(bf16x3, wide, few, k, op)
                    if p is None:
                        continue
                    taken += 1
                    waves, chunks, steps = p
                    # HIP refuses 2^32 threads or more along an axis
                    assert (wide + 31) // 32 * waves * 64 < 1 << 32, (wide, few, k)
                    assert waves in (8, 16) and chunks <= 65535
                    assert steps * chunks >= k // 32 and steps * (chunks - 1) < max(1, k // 32), (wide, few, k)
    assert taken > 20


# Measured with and without the kernel, operands from memory and from the caches: slower by 10 % to four times.
SERVED_FASTER_BY_TILES = [
    (False, "TN", 1024, 16, 1024), (False, "TN", 1024, 16, 2048), (False, "TN", 2048, 1, 4096), (False, "NN", 1024, 8, 4096),
    (False, "TN", 1024, 32, 1024), (False, "TN", 10000, 16, 4096), (False, "NN", 12500, 16, 8192),
    (False, "TN", 65536, 16, 512), (False, "NN", 65536, 16, 1024), (False, "TN", 65536, 32, 128),
    (False, "TN", 1 << 20, 1, 16), (False, "TN", 1 << 20, 16, 4), (False, "NN", 1 << 20, 32, 4),
    (True, "TN", 1024, 16, 2048), (True, "TN", 1024, 32, 4096), (True, "NN", 1024, 32, 2048),
    (True, "TN", 1 << 20, 32, 16), (True, "NN", 1 << 18, 24, 4), (True, "NN", 1 << 20, 32, 128),
    (False, "NN", 1 << 18, 16, 256)]
# ... and faster by 10 % to half
SERVED_FASTER_HERE = [
    (False, "TN", 8192, 16, 8192), (False, "TN", 1024, 16, 256), (False, "NN", 2048, 8, 1024), (False, "TN", 8192, 32, 1024),
    (False, "TN", 10000, 16, 256), (False, "NN", 16384, 1, 1), (False, "TN", 20000, 16, 256), (False, "TN", 12000, 30, 777),
    (True, "TN", 8192, 16, 8192), (True, "TN", 16384, 32, 8192), (True, "NN", 1 << 20, 16, 64), (True, "TN", 1024, 32, 256),
    (True, "TN", 65536, 16, 4096), (True, "NN", 20000, 32, 1024)]


@pytest.mark.parametrize("bf16x3,op,wide,few,k", SERVED_FASTER_BY_TILES)
def test_products_that_the_tiled_kernels_serve_faster_go_to_them(plan, bf16x3, op, wide, few, k):
    assert plan(bf16x3, wide, few, k, op) is None


@pytest.mark.parametrize("bf16x3,op,wide,few,k", SERVED_FASTER_HERE)
def test_products_that_the_narrow_kernel_serves_faster_stay(plan, bf16x3, op, wide, few, k):
    assert plan(bf16x3, wide, few, k, op) is not None


@pytest.mark.parametrize("bf16x3", [False, True])
def test_a_second_workgroup_fits_on_a_cu_where_there_is_one(plan, bf16x3):
    for wide, waves in ((1024, 16), (8192, 16), (8193, 8), (12000, 8), (16384, 8)):
        assert plan(bf16x3, wide, 16, 256)[0] == waves
