"""Results of at most 32 rows or columns: the kernel that reads the large operand once.
Edges: a last tile that ends inside a tile of 32, one and two blocks of the narrow side, K below
a step, inside one and split over workgroups.  NaN between and behind the matrices must not
reach a result; |x| <= 30, so one plane holds the values and every sum is exact."""
import numpy as np
import pytest

from gpu_util import N, T, oracle_gemm, run_gemm
from test_gpu_ragged_k import FP16TCEC, TF32TCEC, _padded_ints

pytestmark = pytest.mark.gpu


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
