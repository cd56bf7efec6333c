"""Results of at most 32 rows or columns: the kernel that reads the large operand once.
Edges: a last tile that ends inside a tile of 32, one and two blocks of the narrow side, K below
a step and inside one.  First without correction terms (NaN between and behind the matrices must not
reach a result; |x| <= 30, so one plane holds the values and every sum is exact), then with them."""
import numpy as np
import pytest

from cumpsgemm_amd import inputs
from gpu_util import N, T, make_operand, oracle_gemm, rel_diff, run_gemm
from test_gpu_ragged_k import FP16TCEC, TF32TCEC, _padded_ints

pytestmark = pytest.mark.gpu
FP32 = 12


@pytest.mark.parametrize("mode", [FP16TCEC, TF32TCEC])
@pytest.mark.parametrize("opa,opb", [(N, N), (T, N), (N, T), (T, T)])
def test_narrow_results_are_exact_on_integers(O, handle, dev, mode, opa, opb):
    rng = np.random.default_rng(5)
    for wide, few, k in ((1024, 1, 1), (1025, 16, 33), (1055, 17, 513), (1100, 32, 95), (1056, 5, 4127)):
        for m, n in ((wide, few), (few, wide)):
            a, lda = _padded_ints(rng, opa, m, k, 3, False)
            b, ldb = _padded_ints(rng, opb, k, n, 1, False)
            beta = float(rng.integers(0, 2))
            c0 = rng.integers(-9, 10, m * n).astype(np.float32)
            c, st = run_gemm(handle, dev, mode, opa, opb, m, n, k, 1.0, a, lda, b, ldb, beta, c0.copy(), m, False)
            assert st == 0
            co = oracle_gemm(O, mode, opa, opb, m, n, k, 1.0, a, lda, b, ldb, beta, c0.copy(), m)
            assert np.array_equal(c, co), (m, n, k, beta)


# wide, few, K, parts of K: the smallest sizes, both block counts, a last tile that shares rows, K with and without a
# partial step, 8 waves (more workgroups than CUs), K split over workgroups with a partial step in the last part
FORMS = [(1024, 1, 7, 1), (1055, 16, 256, 1), (1100, 17, 95, 1), (2049, 32, 513, 1), (8200, 17, 40, 1), (16390, 5, 65, 1),
         (1024, 3, 16417, 8), (1030, 16, 16384, 8)]


@pytest.mark.parametrize("mode", [FP16TCEC, TF32TCEC])
@pytest.mark.parametrize("opa,opb", [(N, N), (T, N), (N, T), (T, T)])
@pytest.mark.parametrize("wide,few,k,parts", FORMS)
def test_narrow_results_with_correction_terms(O, handle, dev, monkeypatch, mode, opa, opb, wide, few, k, parts):
    """Operands that fill every plane, alpha, beta and a padded C; the module id says which kernel ran."""
    for m, n in ((wide, few), (few, wide)):
        big_kc = (opa == T) if m == wide else (opb == N)
        if parts > 1 and ((mode == FP16TCEC and big_kc) or (mode == FP16TCEC and wide % 32)):
            continue                                   # (served by the tiled kernels)
        a, lda = make_operand(inputs.uniform, 71, opa, m, k, 1)
        b, ldb = make_operand(inputs.uniform, 72, opb, k, n, 2)
        ldc = m + 3
        c0 = inputs.uniform(73, ldc * n)
        c, st, mid = run_gemm(handle, dev, mode, opa, opb, m, n, k, 0.75, a, lda, b, ldb, -0.5, c0, ldc, False,
                              want_module_id=True)
        assert st == 0 and mid == (5 if parts == 1 else 105), mid
        ref = O.gemm_fp64(opa, opb, m, n, k, 0.75, a, lda, b, ldb, -0.5, c0, ldc)
        cf = oracle_gemm(O, FP32, opa, opb, m, n, k, 0.75, a, lda, b, ldb, -0.5, c0, ldc)
        co = oracle_gemm(O, mode, opa, opb, m, n, k, 0.75, a, lda, b, ldb, -0.5, c0, ldc)
        # (bars as for the tiled kernels: twice FP32's error; the same products in another order)
        assert O.residual(ref, c, m, n, ldc) <= 2.0 * O.residual(ref, cf, m, n, ldc) + 2.0 ** -24
        assert rel_diff(c, co, m, n, ldc) <= 4 * 2.0 ** -24 * np.sqrt(k)
        assert np.array_equal(c.reshape(n, ldc)[:, m:], c0.reshape(n, ldc)[:, m:])


def test_tiled_kernels_report_their_own_ids(handle, dev, monkeypatch):
    monkeypatch.setenv("CUMPSGEMM_KWAVES", "0")   # (what the narrow kernel leaves would be a small product's: id 6)
    a, b, c0 = inputs.uniform(1, 1024 * 64), inputs.uniform(2, 64 * 16), np.zeros(1024 * 16, np.float32)
    ids = []
    for off in (None, "1"):
        if off:
            monkeypatch.setenv("CUMPSGEMM_NO_NARROW", off)
        ids.append(run_gemm(handle, dev, FP16TCEC, T, N, 1024, 16, 64, 1.0, a, 64, b, 64, 0.0, c0, 1024, False,
                            want_module_id=True)[2])
    assert ids[0] == 5 and ids[1] % 100 < 5
