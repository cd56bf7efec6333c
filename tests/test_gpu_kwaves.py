"""Small products: the kernel whose waves share out K.  Edges: tiles that end at the edge of C, that
start inside the one before and that are larger than C, fewer K-steps than waves, a K that ends inside a
step in each of the waves.  Once with integers and NaN between and behind the matrices (exact), once with
operands that fill every plane."""
import numpy as np
import pytest

from cumpsgemm_amd import inputs
from gpu_util import C, N, T, launched_kernels, make_operand, oracle_gemm, rel_diff, run_gemm
from test_gpu_ragged_k import FP16TC, FP16TCEC, TF32TC, TF32TCEC, _padded_ints

pytestmark = pytest.mark.gpu
FP32, AUTO, SCALING = 12, 9, 11
KWAVES = 6  # module id

LAYOUTS = [(False, N, N), (False, T, N), (False, N, T), (False, T, T), (True, N, N), (True, C, N), (True, N, C), (True, T, T)]
# (form 1: 64 x 64, four waves, 2, 3, 4: 32 x 32, eight, four, one; complex 32 x 32, 1: four, 2: eight; 32 K-values a step)
SIZES = [(64, 64, 1), (65, 129, 31), (70, 100, 33), (127, 64, 128), (96, 65, 160), (129, 70, 257), (64, 130, 995), (200, 90, 64)]
NARROWER = [(1, 1, 40), (31, 5, 33), (40, 17, 300)]  # than a tile: K-contiguous operands only


def _sizes(opa, opb):
    return SIZES + [s for s in NARROWER if opa != N and opb == N]


@pytest.mark.parametrize("mode", [FP16TCEC, TF32TCEC, FP16TC, TF32TC])
@pytest.mark.parametrize("cplx,opa,opb", LAYOUTS)
@pytest.mark.parametrize("form", [1, 2, 3, 4])
def test_small_products_are_exact_on_integers(O, handle, dev, monkeypatch, mode, cplx, opa, opb, form):
    monkeypatch.setenv("CUMPSGEMM_KWAVES", str(form))
    rng = np.random.default_rng(5)
    served = 0
    for m, n, k in _sizes(opa, opb):
        a, lda = _padded_ints(rng, opa, m, k, 3, cplx)
        b, ldb = _padded_ints(rng, opb, k, n, 1, cplx)
        beta = float(rng.integers(0, 2))
        c0 = rng.integers(-9, 10, m * n).astype(np.complex64 if cplx else np.float32)
        c, st, mid = run_gemm(handle, dev, mode, opa, opb, m, n, k, 1.0, a, lda, b, ldb, beta, c0.copy(), m, cplx,
                              want_module_id=True)
        assert st == 0
        served += mid == KWAVES
        # |x| <= 30: one plane holds the values, every partial sum is an integer below 2^24
        co = oracle_gemm(O, mode, opa, opb, m, n, k, 1.0, a, lda, b, ldb, beta, c0.copy(), m)
        assert np.array_equal(c, co), (m, n, k, beta)
    forms = 4 if not cplx else 1 if mode == TF32TCEC else 2
    assert served == (len(_sizes(opa, opb)) if form <= forms else 0)


@pytest.mark.parametrize("mode", [FP16TCEC, TF32TCEC, FP16TC, TF32TC])
@pytest.mark.parametrize("cplx,opa,opb,m,n,k", [(False, N, N, 512, 512, 512), (False, N, T, 128, 128, 128),
                                                (False, T, T, 1000, 900, 777), (True, N, T, 256, 256, 256),
                                                (True, C, N, 512, 512, 512)])
def test_small_products_come_here_and_say_so(handle, dev, mode, cplx, opa, opb, m, n, k):
    """Without any tuning variable: the rule takes them, the module id names the kernel that ran."""
    gen = inputs.complex_normal if cplx else inputs.uniform
    a, lda = make_operand(gen, 1, opa, m, k)
    b, ldb = make_operand(gen, 2, opb, k, n)
    c0 = np.zeros(m * n, a.dtype)
    assert run_gemm(handle, dev, mode, opa, opb, m, n, k, 1.0, a, lda, b, ldb, 0.0, c0, m, cplx,
                    want_module_id=True)[1:] == (0, KWAVES)


@pytest.mark.parametrize("mode", [FP16TCEC, TF32TCEC])
@pytest.mark.parametrize("cplx,opa,opb", LAYOUTS)
@pytest.mark.parametrize("form", [1, 2, 3, 4])
def test_small_products_with_correction_terms(O, handle, dev, monkeypatch, mode, cplx, opa, opb, form):
    """Batches with gaps, alpha, beta, a padded C."""
    monkeypatch.setenv("CUMPSGEMM_KWAVES", str(form))
    gen = inputs.complex_normal if cplx else inputs.uniform
    alpha, beta = (0.75 - 0.5j, -0.5 + 0.25j) if cplx else (0.75, -0.5)
    for m, n, k, batch in ((64, 64, 500, 1), (101, 77, 129, 3), (130, 66, 1000, 2)):
        ra, ca = (m, k) if opa == N else (k, m)
        rb, cb = (k, n) if opb == N else (n, k)
        lda, ldb, ldc = ra + 1, rb + 2, m + 3
        sa, sb, sc = lda * ca + 5, ldb * cb + 3, ldc * n + 7
        a, b, c0 = gen(81, sa * batch), gen(82, sb * batch), gen(83, sc * batch)
        da, db, dc = dev.up(a), dev.up(b), dev.up(c0)
        st = handle.gemm_strided_batch(opa, opb, m, n, k, alpha, da, lda, sa, db, ldb, sb, beta, dc, ldc, sc, batch, mode,
                                       cplx=cplx)
        assert st == 0
        out = dev.down(dc, np.complex64 if cplx else np.float32)
        for i in range(batch):
            ai, bi, ci, x = a[i * sa:][:lda * ca], b[i * sb:][:ldb * cb], c0[i * sc:][:ldc * n], out[i * sc:][:ldc * n]
            ref = O.gemm_fp64(opa, opb, m, n, k, alpha, ai, lda, bi, ldb, beta, ci, ldc)
            cf = oracle_gemm(O, FP32, opa, opb, m, n, k, alpha, ai, lda, bi, ldb, beta, ci, ldc)
            co = oracle_gemm(O, mode, opa, opb, m, n, k, alpha, ai, lda, bi, ldb, beta, ci, ldc)
            # (bars as for the tiled kernels: twice FP32's error; the same products in another order)
            assert O.residual(ref, x, m, n, ldc) <= 2.0 * O.residual(ref, cf, m, n, ldc) + 2.0 ** -24
            assert rel_diff(x, co, m, n, ldc) <= 4 * 2.0 ** -24 * np.sqrt(k)
            assert np.array_equal(x.reshape(n, ldc)[:, m:], ci.reshape(n, ldc)[:, m:])
            assert np.array_equal(out[i * sc + ldc * n:(i + 1) * sc], c0[i * sc + ldc * n:(i + 1) * sc])


@pytest.mark.parametrize("mode,exponent", [(SCALING, 40), (AUTO, 40), (AUTO, 0)])
@pytest.mark.parametrize("cplx,opa,opb", LAYOUTS)
def test_small_products_scaled_and_gated(handle, dev, monkeypatch, mode, exponent, cplx, opa, opb):
    """Integers times 2^40 (A) and 2^-40 (B): exact in either mode that AUTO may decide for; with the form forced the
    result is that of the tiled kernels bit for bit."""
    rng = np.random.default_rng(8)
    for m, n, k in ((64, 64, 31), (130, 100, 127), (96, 70, 300)):
        a, lda = _padded_ints(rng, opa, m, k, 0, cplx)
        b, ldb = _padded_ints(rng, opb, k, n, 0, cplx)
        s = np.float32(2.0 ** exponent)
        outs = []
        for form in ("1", "2", "3", "4", "0"):
            monkeypatch.setenv("CUMPSGEMM_KWAVES", form)
            da, db, dc = dev.up(a * s), dev.up(b / s), dev.up(np.full(m * n, np.nan, np.complex64 if cplx else np.float32))
            st, _ = handle.gemm_pipeline(opa, opb, m, n, k, 1.0, da, lda, db, ldb, 0.0, dc, m, mode, cplx=cplx)
            assert st == 0
            outs.append(dev.down(dc, np.complex64 if cplx else np.float32))
        assert np.isfinite(outs[0].view(np.float32)).all()
        assert all(np.array_equal(x, outs[-1]) for x in outs[:-1])


@pytest.mark.parametrize("mode,scaled_b,want", [(SCALING, True, FP16TCEC), (AUTO, False, FP16TCEC), (AUTO, True, FP16TCEC),
                                                (AUTO, None, TF32TCEC)])
@pytest.mark.parametrize("cplx,opa,opb,form", [(*layout, form) for layout in LAYOUTS for form in ((1, 2) if layout[0] else (1, 2, 3, 4))])
def test_small_products_scaled_and_gated_with_correction_terms(handle, dev, monkeypatch, mode, scaled_b, want, cplx, opa,
                                                               opb, form):
    """Operands that fill every plane: with the form forced a pipeline call gives, bit for bit, what the decided mode
    gives for operands scaled beforehand -- which is checked against the oracle above, and whose module id says that
    the form ran.  (K < 256: no tiled plan splits it, so each of AUTO's candidates takes the form if it has it.)"""
    monkeypatch.setenv("CUMPSGEMM_KWAVES", str(form))
    gen = inputs.complex_normal if cplx else inputs.uniform
    dtype = np.complex64 if cplx else np.float32
    handle.set_exp_stats_params(0.0, 2.0 ** -15, 0.1)
    try:
        for m, n, k in ((130, 100, 250), (66, 129, 95)):
            a, lda = make_operand(gen, 91, opa, m, k)
            b, ldb = make_operand(gen, 92, opb, k, n)
            if scaled_b:
                b *= np.float32(2.0 ** -40)       # every element below fp16's range
            elif scaled_b is None:
                b[::2] *= np.float32(2.0 ** -60)  # too far from the others for any scaling
            c0 = gen(93, m * n)
            da, db, dc = dev.up(a), dev.up(b), dev.up(c0)
            st, (_, _, flag) = handle.gemm_pipeline(opa, opb, m, n, k, 0.75, da, lda, db, ldb, -0.5, dc, m, mode, cplx=cplx)
            assert st == 0 and handle.get_dynamic_launch_flag(flag) & 31 == want
            got = dev.down(dc, dtype)

            def factor(x):  # 2^14 over the largest element's power of two
                return np.float32(2.0 ** (14 - np.floor(np.log2(np.abs(x.view(np.float32)).max()))))
            sa, sb = factor(a) if mode == SCALING else np.float32(1), factor(b) if scaled_b else np.float32(1)
            ref, st, mid = run_gemm(handle, dev, want, opa, opb, m, n, k, 0.75 / float(sa * sb), a * sa, lda, b * sb, ldb,
                                    -0.5, c0, m, cplx, want_module_id=True)
            assert st == 0 and (mid == KWAVES) == (not cplx or form == 1 or want == FP16TCEC)
            assert np.array_equal(got.view(np.uint32), ref.view(np.uint32)), (m, n, k)
    finally:
        handle.set_exp_stats_params(0.0, 2.0 ** -15, 0.0)


def test_no_kslice_groups_leaves_small_products_alone(handle, dev, monkeypatch):
    """CUMPSGEMM_NO_KSLICE_GROUPS chooses between two forms of the tiled kernel, nothing else."""
    a, b, c0 = inputs.uniform(1, 512 * 512), inputs.uniform(2, 512 * 512), np.zeros(512 * 512, np.float32)
    monkeypatch.setenv("CUMPSGEMM_NO_KSLICE_GROUPS", "1")
    assert run_gemm(handle, dev, FP16TCEC, N, N, 512, 512, 512, 1.0, a, 512, b, 512, 0.0, c0, 512, False,
                    want_module_id=True)[1:] == (0, KWAVES)


def test_auto_compares_small_products_with_the_tiled_plan_that_runs(handle, dev, monkeypatch):
    """AUTO's FP16TCEC candidate where its own tiled plan would split K, but cannot, as the bf16x3 plan does not: the
    unsplit plan is the one that it would run, and it is slower than the small-product kernel."""
    m, n, k = 795, 1259, 1765
    a, b = inputs.uniform(1, m * k), inputs.uniform(2, k * n)
    da, db = dev.up(a), dev.up(b)
    outs = []
    handle.set_exp_stats_params(0.0, 2.0 ** -15, 0.1)  # FP16TCEC for these operands
    try:
        for form in (None, "2"):
            if form:
                monkeypatch.setenv("CUMPSGEMM_KWAVES", form)
            dc = dev.up(np.zeros(m * n, np.float32))
            st, (_, _, flag) = handle.gemm_pipeline(N, N, m, n, k, 1.0, da, m, db, k, 0.0, dc, m, AUTO)
            assert st == 0 and handle.get_dynamic_launch_flag(flag) == FP16TCEC
            outs.append(dev.down(dc))
    finally:
        handle.set_exp_stats_params(0.0, 2.0 ** -15, 0.0)
    assert np.array_equal(outs[0], outs[1])  # (a tiled kernel adds in another order)


@pytest.mark.parametrize("mode", [FP16TCEC, TF32TC, SCALING])
@pytest.mark.parametrize("opa,opb", [(N, N), (C, N), (N, T), (T, C)])
def test_complex_two_wave_groups_are_exact_on_integers(O, handle, dev, monkeypatch, mode, opa, opb):
    """The tiled kernel that complex products of a few tiles take otherwise, its operands loaded two steps
    ahead: one to six K-steps, with and without a partial one, tiles at the edge and larger than C."""
    monkeypatch.setenv("CUMPSGEMM_KWAVES", "0")
    rng = np.random.default_rng(6)
    for k in (31, 32, 33, 64, 65, 96, 97, 128, 129, 160, 190, 995):
        for m, n in ((64, 128), (131, 70), (37, 9)):
            a, lda = _padded_ints(rng, opa, m, k, 3, True)
            b, ldb = _padded_ints(rng, opb, k, n, 1, True)
            beta = float(rng.integers(0, 2))
            c0 = rng.integers(-9, 10, m * n).astype(np.complex64)
            c, st = run_gemm(handle, dev, mode, opa, opb, m, n, k, 1.0, a, lda, b, ldb, beta,
                             c0.copy(), m, True)
            assert st == 0
            co = oracle_gemm(O, FP16TCEC if mode == SCALING else mode, opa, opb, m, n, k, 1.0, a, lda, b, ldb, beta,
                             c0.copy(), m)
            assert np.array_equal(c, co), (m, n, k, beta)


@pytest.mark.parametrize("mode", [FP16TCEC, FP16TC, TF32TC])
@pytest.mark.parametrize("cplx,opa,opb,m,n,k", [(False, N, N, 1100, 1000, 290), (False, T, N, 1090, 1030, 257),
                                                (False, N, T, 1153, 1000, 161), (True, N, N, 580, 540, 290),
                                                (True, N, C, 577, 545, 130)])
def test_more_tiles_than_cus_are_exact_on_integers(O, handle, dev, monkeypatch, mode, cplx, opa, opb, m, n, k):
    """Two workgroups of the 64 x 64 (complex 32 x 32) form on one CU."""
    monkeypatch.setenv("CUMPSGEMM_KWAVES", "1")
    rng = np.random.default_rng(9)
    a, lda = _padded_ints(rng, opa, m, k, 3, cplx)
    b, ldb = _padded_ints(rng, opb, k, n, 1, cplx)
    c0 = rng.integers(-9, 10, m * n).astype(np.complex64 if cplx else np.float32)
    c, st, mid = run_gemm(handle, dev, mode, opa, opb, m, n, k, 1.0, a, lda, b, ldb, 1.0, c0.copy(), m, cplx,
                          want_module_id=True)
    assert (st, mid) == (0, KWAVES)
    # |x| <= 30: every partial sum is an integer below 2^24
    assert np.array_equal(c, oracle_gemm(O, mode, opa, opb, m, n, k, 1.0, a, lda, b, ldb, 1.0, c0.copy(), m))


@pytest.mark.parametrize("mode", [FP16TCEC, FP16TC, TF32TC])
@pytest.mark.parametrize("cplx,opa,opb", LAYOUTS)
def test_forms_for_one_workgroup_on_a_cu(O, handle, dev, monkeypatch, mode, cplx, opa, opb):
    """Form 5: real FP16TCEC 64 x 64 with two sets of fragments, complex 64 x 32."""
    monkeypatch.setenv("CUMPSGEMM_KWAVES", "5")
    rng = np.random.default_rng(10)
    for m, n, k in _sizes(opa, opb):
        a, lda = _padded_ints(rng, opa, m, k, 3, cplx)
        b, ldb = _padded_ints(rng, opb, k, n, 1, cplx)
        c0 = rng.integers(-9, 10, m * n).astype(np.complex64 if cplx else np.float32)
        c, st, mid = run_gemm(handle, dev, mode, opa, opb, m, n, k, 1.0, a, lda, b, ldb, 1.0, c0.copy(), m, cplx,
                              want_module_id=True)
        assert st == 0 and (mid == KWAVES) == (cplx or mode == FP16TCEC)
        # (as above: every partial sum is an integer below 2^24)
        assert np.array_equal(c, oracle_gemm(O, mode, opa, opb, m, n, k, 1.0, a, lda, b, ldb, 1.0, c0.copy(), m)), (m, n, k)
    if mode == FP16TCEC:
        test_small_products_with_correction_terms(O, handle, dev, monkeypatch, mode, cplx, opa, opb, 5)
        for args in ((SCALING, True, FP16TCEC), (AUTO, True, FP16TCEC)):
            test_small_products_scaled_and_gated_with_correction_terms(handle, dev, monkeypatch, *args, cplx, opa, opb, 5)


def _auto_call(handle, dev, opa, opb, m, n, k, batch, cplx, decided, before_reference, after_reference):
    """(call, C on the device, the explicit mode's result of the same call): padded, with gaps, beta != 0.
    `decided`: what the operands make AUTO decide for."""
    gen = inputs.complex_normal if cplx else inputs.uniform
    ra, ca = (m, k) if opa == N else (k, m)
    rb, cb = (k, n) if opb == N else (n, k)
    lda, ldb, ldc = ra + 1, rb + 2, m + 3
    sa, sb, sc = lda * ca + 5, ldb * cb + 3, ldc * n + 7
    a, b, c0 = gen(94, sa * batch), gen(95, sb * batch), gen(96, sc * batch)
    if decided == TF32TCEC:
        b[::2] *= np.float32(2.0 ** -60)
    da, db, dc, dr = dev.up(a), dev.up(b), dev.up(c0), dev.up(c0)

    def call():
        st, ids = handle.gemm_pipeline(opa, opb, m, n, k, 0.75, da, lda, db, ldb, -0.5, dc, ldc, AUTO, cplx=cplx, stridea=sa,
                                       strideb=sb, stridec=sc, batch=batch)
        assert st == 0
        return ids[2]
    before_reference()
    st = handle.gemm_strided_batch(opa, opb, m, n, k, 0.75, da, lda, sa, db, ldb, sb, -0.5, dr, ldc, sc, batch, decided, cplx=cplx)
    after_reference()
    assert st == 0
    return call, dc, dr


# as dispatched (then: the form that the shared launch takes), and every form that both candidates have forced; K = 2000:
# bf16x3's tiled plan splits K and would prepare C
@pytest.mark.parametrize("decided", [FP16TCEC, TF32TCEC])
@pytest.mark.parametrize("cplx,m,n,k,batch,form,one_launch", [
    (False, 512, 512, 512, 1, "as dispatched 2", True), (False, 130, 100, 250, 3, "1", True), (False, 101, 77, 129, 5, "2", True),
    (False, 66, 129, 95, 3, "3", True), (False, 130, 66, 250, 4, "4", True), (True, 256, 256, 256, 1, "as dispatched 1", True),
    (True, 101, 77, 129, 3, "1", True), (True, 577, 545, 1000, 1, "1", False), (True, 577, 545, 2000, 1, "1", False),
    (True, 300, 290, 1000, 4, "1", False)])
def test_auto_in_one_launch_or_two(torch_gpu, handle, dev, monkeypatch, decided, cplx, m, n, k, batch, form, one_launch):
    """Which kernels run, and that the result is the decided mode's bit for bit, gaps of C included."""
    forced, form = not form.startswith("as"), form[-1]

    def force():
        monkeypatch.setenv("CUMPSGEMM_KWAVES", form)

    def release():
        if not forced:
            monkeypatch.delenv("CUMPSGEMM_KWAVES")
    if forced:
        force()
    handle.set_exp_stats_params(0.0, 2.0 ** -15, 0.1)
    try:
        for opa, opb in ((N, N), (C if cplx else T, N), (N, T), (T, C if cplx else T)):
            call, dc, dr = _auto_call(handle, dev, opa, opb, m, n, k, batch, cplx, decided, force, release)
            assert handle.get_dynamic_launch_flag(call()) & 31 == decided
            out = np.complex64 if cplx else np.float32
            assert np.array_equal(dev.down(dc, out).view(np.uint32), dev.down(dr, out).view(np.uint32)), (opa, opb)
            ran = [(name, grid) for name, grid in launched_kernels(torch_gpu, handle, call) if "exp_stats" not in name]
            assert len(ran) == (1 if one_launch else 2), ran
            assert all(("kwaves_either_gemm" if one_launch else "kwaves_gemm") in name for name, _ in ran), ran
            bm = 64 if not cplx and form == "1" else 32
            assert all(grid[0] == -(-m // bm) * -(-n // bm) * batch for _, grid in ran), ran
    finally:
        handle.set_exp_stats_params(0.0, 2.0 ** -15, 0.0)
