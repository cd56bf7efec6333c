"""The rule that sends small products to their kernel (csrc/kwaves_rule.hpp), compiled for the host: what
it takes, the kernel can serve and a launch can hold; nothing else reaches the kernel, whatever is asked for."""
import ctypes
import itertools
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "cumpsgemm_amd", "csrc")
CUS = 256
u64 = ctypes.c_uint64


@pytest.fixture(scope="module")
def rule(tmp_path_factory):
    d = tmp_path_factory.mktemp("rule")
    (d / "rule.cpp").write_text("""
        #include "kwaves_rule.hpp"
        using namespace cumpsgemm_amd;
        extern "C" int form(int prec, int cplx, int a_kc, int b_kc, uint64_t m, uint64_t n, uint64_t k, uint64_t batch,
                            uint64_t lda, uint64_t ldb, double steps, int split, int asked, int *tile) {
          const KWavesProblem p{cplx != 0, a_kc != 0, b_kc != 0, m, n, k, batch, lda, ldb};
          const int f = choose_kwaves_form(prec, p, 256, steps, split != 0, asked);
          if (f >= 0) {
            const KWavesForm &x = kwaves_model(prec, p.cplx).form[f];
            tile[0] = x.bm, tile[1] = x.bn, tile[2] = x.waves;
          }
          return f;
        }
        extern "C" int either(int cplx, int a_kc, int b_kc, uint64_t m, uint64_t n, uint64_t k, uint64_t batch, uint64_t lda,
                              uint64_t ldb, int form_bf16, int form_fp16) {
          return choose_kwaves_either_form({cplx != 0, a_kc != 0, b_kc != 0, m, n, k, batch, lda, ldb}, 256, form_bf16,
                                           form_fp16);
        }""")
    so = d / "rule.so"
    subprocess.check_call(["g++", "-std=c++17", "-shared", "-fPIC", "-I", CSRC, "-o", str(so), str(d / "rule.cpp")])
    lib = ctypes.CDLL(str(so))

    def call(prec, cplx, op, m, n, k, batch=1, pad=0, steps=1e9, split=False, asked=-1):
        """(form, bm, bn, waves) or None"""
        lda, ldb = (m if op[0] == "N" else k) + pad, (k if op[1] == "N" else n) + pad
        tile = (ctypes.c_int * 3)()
        f = lib.form(prec, int(cplx), int(op[0] != "N"), int(op[1] == "N"), u64(m), u64(n), u64(k), u64(batch), u64(lda),
                     u64(ldb), ctypes.c_double(steps), int(split), asked, tile)
        return (f, *tile) if f >= 0 else None

    def either(cplx, op, m, n, k, batch, form_bf16, form_fp16):
        return lib.either(int(cplx), int(op[0] != "N"), int(op[1] == "N"), u64(m), u64(n), u64(k), u64(batch),
                          u64(m if op[0] == "N" else k), u64(k if op[1] == "N" else n), form_bf16, form_fp16)
    call.either = either
    return call


@pytest.mark.parametrize("asked", [-1, 1, 2, 3, 4])
def test_what_the_rule_takes_can_be_served(rule, asked):
    sizes = (1, 31, 32, 63, 64, 65, 1000, 1 << 20, (1 << 26) + 1, (1 << 31) - 1)
    taken = 0
    for prec, cplx, op in itertools.product(range(4), (False, True), ("NN", "TN", "NT", "TT")):
        for m, n, k, batch, pad in itertools.product(sizes, sizes, (1, 33, 1000, (1 << 31) - 1), (1, 65535), (0, 3)):
            p = rule(prec, cplx, op, m, n, k, batch, pad, asked=asked)
            if p is None:
                continue
            taken += 1
            _, bm, bn, waves = p
            # a row-contiguous operand's tile lies inside the matrix
            assert (op[0] != "N" or m >= bm) and (op[1] == "N" or n >= bn)
            # HIP refuses 2^32 threads or more along an axis; byte offsets inside a tile are 31 bits
            assert -(-m // bm) * -(-n // bn) * batch * waves * 64 < 1 << 32
            es = 8 if cplx else 4
            lda, ldb = (m if op[0] == "N" else k) + pad, (k if op[1] == "N" else n) + pad
            for kc, rows, ld in ((op[0] != "N", bm, lda), (op[1] == "N", bn, ldb)):
                assert ((rows - 1) * ld + 32 if kc else 31 * ld + rows) * es < 1 << 31
    assert taken > 1000


def test_the_rule_compares_with_the_tiled_plan(rule):
    for prec, cplx in itertools.product(range(4), (False, True)):
        assert rule(prec, cplx, "NN", 512, 512, 512) is not None                       # the tiled kernels take for ever
        assert rule(prec, cplx, "NN", 512, 512, 512, steps=0.0) is None                # no time at all
        assert rule(prec, cplx, "NN", 512, 512, 512, asked=0) is None                  # switched off
        assert rule(prec, cplx, "NN", 512, 512, 0) is None                             # nothing to multiply
        assert rule(prec, cplx, "NN", 8192, 8192, 8192) is None                        # too large for small tiles


@pytest.mark.parametrize("prec,op,m,n,k,batch,steps,split,waves", [
    (1, "NN", 2560, 586, 224, 1, 4.5, False, 4), (0, "TN", 637, 64, 256, 34, 4.9, False, 4),
    (0, "TT", 64, 40, 243, 352, 4.9, False, 4), (0, "NN", 736, 1349, 8128, 1, 77.7, True, None),
    (0, "NN", 1920, 544, 4354, 1, 47.1, True, None)])
def test_eight_waves_on_a_tile_in_one_round_only(rule, prec, op, m, n, k, batch, steps, split, waves):
    """Products whose eight-wave workgroups a chip of 256 CUs cannot hold at once (`steps`: the tiled plan's cost):
    measured slower than with four waves, or than tiled where K is long and the tiled plan splits it."""
    p = rule(prec, False, op, m, n, k, batch, steps=steps, split=split)
    assert (p and p[3]) == waves
    for m, n in itertools.product((512, 736, 1024, 1333), (512, 1024, 1536)):
        p = rule(prec, False, op, m, n, k, steps=1e3, split=split)
        assert p is None or p[3] != 8 or -(-m // 32) * -(-n // 32) <= 2 * CUS


@pytest.mark.parametrize("prec,m,n,k,steps", [(1, 1090, 256, 3360, 15.4), (1, 2549, 112, 2560, 12.6), (0, 528, 528, 2880, 13.7)])
def test_a_long_k_of_two_row_contiguous_operands_is_split(rule, prec, m, n, k, steps):
    """Two eight-wave workgroups on a CU, K as long and split by the tiled plan (`steps`: its cost): measured slower."""
    assert rule(prec, False, "NT", m, n, k, steps=steps, split=True) is None
    for op, kk, split in (("TN", k, True), ("NT", 1500, True), ("NT", k, False)):
        assert rule(prec, False, op, m, n, kk, steps=2 * steps, split=split) is not None


@pytest.mark.parametrize("op", ["NN", "TN", "NT", "TT"])
@pytest.mark.parametrize("cplx", [False, True])
def test_one_launch_for_both_candidates_of_auto(rule, cplx, op):
    """It takes the form of one of the two, which can serve the product in either precision; none where a candidate is
    not here or where FP16TCEC would lose its second workgroup per CU."""
    taken = 0
    sizes = (1, 31, 32, 64, 100, 512, 640, 1200, 1 << 26, (1 << 31) - 1)
    for m, n, k, batch in itertools.product(sizes, sizes, (1, 100, 1000, (1 << 31) - 1), (1, 65535)):
        a, b = rule(2, cplx, op, m, n, k, batch), rule(0, cplx, op, m, n, k, batch)
        form = rule.either(cplx, op, m, n, k, batch, a[0] if a else -1, b[0] if b else -1)
        if form < 0:
            continue
        taken += 1
        assert form in (a[0], b[0])
        tiles = [rule(prec, cplx, op, m, n, k, batch, asked=form + 1) for prec in (2, 0)]
        assert tiles[0] is not None and tiles[0] == tiles[1]
    assert taken > 50
    assert rule.either(cplx, op, 512, 512, 512, 1, 0, -1) == rule.either(cplx, op, 512, 512, 512, 1, -1, 0) == -1
    assert rule.either(cplx, op, 512, 512, 512, 1, 0, 0) == 0
    if cplx:
        assert rule.either(cplx, op, 640, 640, 640, 1, 0, 0) == -1


# (`steps`, `split`: the tiled plan's cost, whether it splits K)
@pytest.mark.parametrize("prec,cplx,op,m,n,k,steps,split,tile", [
    (0, False, "NN", 3968, 173, 2378, 18.86, True, (64, 64, 4)), (0, False, "TT", 1485, 530, 2754, 21.33, True, (64, 64, 4)),
    (0, False, "NT", 310, 1884, 1600, 14.63, True, (64, 64, 4)), (1, True, "NT", 431, 1024, 3798, 30.48, True, (64, 32, 4)),
    (1, True, "NN", 384, 1118, 2033, 23.52, True, (64, 32, 4))])
def test_one_workgroup_on_a_cu_has_the_registers_of_a_simd_to_itself(rule, prec, cplx, op, m, n, k, steps, split, tile):
    """Measured 1.05 - 1.35 times as long on the forms of two waves to a SIMD, or on the kernel taken instead."""
    p = rule(prec, cplx, op, m, n, k, steps=steps, split=split)
    assert p and p[1:] == tile and p[0] == 4
    # never where a CU has a second workgroup, nor for a short K
    for mm, nn in itertools.product((m, 2 * m, 3 * m), (n, 3 * n)):
        q = rule(prec, cplx, op, mm, nn, k, steps=1e3, split=split)
        assert q is None or q[0] != 4 or -(-mm // tile[0]) * -(-nn // tile[1]) <= CUS
    q = rule(prec, cplx, op, m, n, 200, steps=1e3, split=split)
    assert q is None or q[0] != 4


@pytest.mark.parametrize("prec,op,m,n,k,steps", [(3, "TT", 528, 1440, 447, 7.97), (3, "NN", 960, 576, 448, 7.97),
                                                (1, "NN", 768, 768, 203, 4.76), (0, "TT", 208, 2496, 512, 8.85)])
def test_eight_waves_on_a_complex_tile_in_one_round_only(rule, prec, op, m, n, k, steps):
    """More tiles than CUs: measured 1.1 - 1.35 times as long as with four waves."""
    assert rule(prec, True, op, m, n, k, steps=steps) == (0, 32, 32, 4)
    for prec, mm, nn, kk in itertools.product((0, 1, 3), (256, 512, 1024), (300, 512, 2000), (64, 400, 3000)):
        p = rule(prec, True, op, mm, nn, kk, steps=1e3)
        assert p is None or p[3] != 8 or -(-mm // 32) * -(-nn // 32) <= CUS


@pytest.mark.parametrize("prec,op,m,n,k,batch,pad,steps", [
    (3, "NN", 512, 2254, 128, 1, 0, 3.27), (3, "TN", 2891, 416, 100, 1, 4, 3.27), (1, "TN", 4576, 288, 160, 1, 0, 3.68),
    (1, "TT", 96, 96, 96, 117, 4, 2.86), (0, "TT", 608, 2560, 192, 1, 0, 4.09), (0, "NN", 224, 5088, 104, 1, 0, 3.27)])
def test_a_short_k_of_257_to_512_large_tiles_takes_small_ones(rule, prec, op, m, n, k, batch, pad, steps):
    """Measured 1.2 - 1.3 times as long on 64 x 64 tiles as on 32 x 32."""
    assert rule(prec, False, op, m, n, k, batch, pad, steps=steps)[1:3] == (32, 32)


@pytest.mark.parametrize("prec", [0, 1, 3])
def test_two_rounds_of_large_tiles_at_most_and_no_third_tile_on_a_cu(rule, prec):
    """64 x 64 tiles, K beyond 512, two workgroups to a CU; `steps`: the tiled kernels are estimated at 1.7 times as long."""
    for op in ("NN", "TN", "NT", "TT"):
        for tiles_m, tiles_n, taken in ((16, 32, True), (19, 27, op == "NT"), (24, 32, op == "NT"), (25, 31, True), (32, 32, True),
                                        (25, 41, False)):
            m, n, rounds = 64 * tiles_m, 64 * tiles_n, 1 if tiles_m * tiles_n <= 2 * CUS else 2
            p = rule(prec, False, op, m, n, 2000, steps={0: 42, 1: 45, 3: 42}[prec] * rounds)
            assert (p and p[:3]) == ((0, 64, 64) if taken else None), (op, tiles_m, tiles_n)
        assert rule(prec, False, op, 64 * 19, 64 * 27, 500, steps=40) is not None


@pytest.mark.parametrize("prec,op,m,n,k,batch,pad,steps", [
    (0, "TN", 53, 265, 411, 608, 0, 49.27), (1, "TT", 320, 320, 320, 159, 0, 52.19), (1, "NT", 128, 128, 128, 331, 0, 9.94),
    (0, "TT", 704, 393, 231, 17, 0, 13.31), (1, "NN", 160, 288, 640, 47, 1, 45.0)])
def test_batches_of_several_rounds_keep_their_large_tiles(rule, prec, op, m, n, k, batch, pad, steps):
    """Measured 0.61 - 0.91 of the tiled time on 64 x 64 tiles."""
    assert rule(prec, False, op, m, n, k, batch, pad, steps=steps)[:3] == (0, 64, 64)
