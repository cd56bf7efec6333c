"""Results narrower than a tile and a K that ends inside a K-step: the kernels read such
operands without branches (the last row or column again, K-values past the end replaced by
zero).  NaN in everything that lies between and behind the matrices -- row padding, the
memory after the last element -- must not reach a result, and small integers must come out
exactly."""
import numpy as np
import pytest

from gpu_util import N, T, C, oracle_gemm, run_gemm, stored_shape

pytestmark = pytest.mark.gpu

FP16TCEC, TF32TCEC, FP16TC, TF32TC = 1, 2, 3, 4


def _padded_ints(rng, op, rows, cols, pad, cplx):
    r, c = stored_shape(op, rows, cols)
    x = np.full((c + 1, r + pad), np.nan + (1j * np.nan if cplx else 0), np.complex64 if cplx else np.float32)
    x[:c, :r] = rng.integers(-30, 31, (c, r))
    if cplx:
        x[:c, :r] += 1j * rng.integers(-30, 31, (c, r))
    return x.reshape(-1), r + pad


@pytest.mark.parametrize("cls", [0, 1, 2, 3, 4])
@pytest.mark.parametrize("cplx,opa,opb,mode", [
    (False, N, N, FP16TCEC), (False, T, N, FP16TCEC), (False, N, T, FP16TCEC), (False, T, T, FP16TCEC),
    (False, N, N, TF32TCEC), (False, T, T, TF32TCEC), (False, N, T, FP16TC), (False, T, N, TF32TC),
    (True, N, N, FP16TCEC), (True, C, T, FP16TCEC), (True, N, C, TF32TCEC), (True, T, N, FP16TC)])
def test_partial_tiles_and_k_steps_read_nothing_but_the_matrices(O, handle, dev, monkeypatch, cls, cplx, opa, opb, mode):
    monkeypatch.setenv("CUMPSGEMM_FORCE_TILE_CLASS", str(cls))
    monkeypatch.setenv("CUMPSGEMM_PACKED", "0")
    rng = np.random.default_rng(3)
    for m, n, k in ((1, 1, 1), (31, 5, 33), (65, 16, 31), (100, 100, 100), (16, 129, 63), (257, 40, 65), (300, 290, 127),
                    (40, 17, 1000)):
        a, lda = _padded_ints(rng, opa, m, k, 3, cplx)
        b, ldb = _padded_ints(rng, opb, k, n, 1, cplx)
        c0 = np.zeros(m * n, np.complex64 if cplx else np.float32)
        c, st = run_gemm(handle, dev, mode, opa, opb, m, n, k, 1.0, a, lda, b, ldb, 0.0, c0, m, cplx)
        assert st == 0
        # |x| <= 30: one plane holds the values, every partial sum is an integer below 2^24
        co = oracle_gemm(O, mode, opa, opb, m, n, k, 1.0, a, lda, b, ldb, 0.0, c0, m)
        assert np.array_equal(c, co), (m, n, k)


@pytest.mark.parametrize("opa,opb", [(N, N), (T, N), (N, T), (T, T)])
def test_scaled_large_tiles_at_edges_and_partial_k_steps(handle, dev, monkeypatch, opa, opb):
    """The 256x128 kernel with the scaling of A and B in it: one tile beyond the edges, moved tiles, K below a step,
    inside one and a step more; integers times 2^40 stay exact, padding and what lies behind are NaN."""
    monkeypatch.setenv("CUMPSGEMM_FORCE_TILE_CLASS", "0")
    monkeypatch.setenv("CUMPSGEMM_PACKED", "0")
    rng = np.random.default_rng(8)
    for m, n, k in ((100, 100, 100), (256, 128, 31), (256, 100, 96), (300, 290, 127), (513, 129, 33)):
        a, lda = _padded_ints(rng, opa, m, k, 3, False)
        b, ldb = _padded_ints(rng, opb, k, n, 1, False)
        s = np.float32(2.0 ** 40)
        da, db, dc = dev.up(a * s), dev.up(b / s), dev.up(np.full(m * n, np.nan, np.float32))
        st, _ = handle.gemm_pipeline(opa, opb, m, n, k, 1.0, da, lda, db, ldb, 0.0, dc, m, 11)  # FP16TCEC_SCALING
        assert st == 0

        def logical(x, op, ld, rows, cols):
            v = x.reshape(-1, ld)[:cols if op == N else rows, :rows if op == N else cols].astype(np.float64)
            return v.T if op == N else v
        want = logical(a, opa, lda, m, k) @ logical(b, opb, ldb, k, n)
        assert np.array_equal(dev.down(dc).reshape(n, m).T, want), (m, n, k)
