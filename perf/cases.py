"""The GEMM calls whose speed this library is kept to: what a program that uses
it for its FP32 / complex64 products has it do, from the smallest calls, where
latency and launches count, to the largest.

`listed()` names the fixed cases, `draw(rng)` makes one more of the same ranges.
A case is a dict of plain values; `prepare` makes the operands on the GPU and the
handle that a program keeps, `run` is one pass through the public entry points
(`cumpsgemm_amd.Handle`), `work` the bytes and matrix-core flops a pass cannot do
without and `tolerance` how far another correct implementation of the same
arithmetic may be from this one.
"""
import math

import torch

import cumpsgemm_amd as cg

OPS = {"N": cg.OP_N, "T": cg.OP_T, "C": cg.OP_C}
MODES = {"FP16TCEC": cg.FP16TCEC, "TF32TCEC": cg.TF32TCEC, "FP16TC": cg.FP16TC, "TF32TC": cg.TF32TC,
         "FP16TCEC_SCALING": cg.FP16TCEC_SCALING, "AUTO": cg.AUTO}
# matrix-core products per multiply-add of the result: the arithmetic that the
# mode stands for (hi*hi + hi*lo + lo*hi; six of the nine bf16 products; one).
# AUTO is asked about operands that it serves with FP16TCEC.
PRODUCTS = {"FP16TCEC": 3, "TF32TCEC": 6, "FP16TC": 1, "TF32TC": 3, "FP16TCEC_SCALING": 3, "AUTO": 3}
# no drawn case asks for more than the largest listed one
MOST_FLOPS = 3 * 2.0 * 8192 ** 3
MOST_BYTES = 4.4e9


def _gemm(m, n, k, mode="FP16TCEC", op="NN", cplx=False, batch=1, beta=0.0, pad=0, data="uniform"):
    return {"kind": "gemm", "m": m, "n": n, "k": k, "mode": mode, "op": op, "cplx": cplx, "batch": batch, "beta": beta,
            "pad": pad, "data": data}


def _gate(rows, cplx=True, wide=False):
    return {"kind": "gate", "rows": rows, "cplx": cplx, "wide": wide}


def listed():
    return [
        # the smallest calls: one launch of a few workgroups, host path and latency
        dict(name="sgemm_128", **_gemm(128, 128, 128)),
        # an ordinary square product (fewer large tiles than the chip has CUs)
        dict(name="sgemm_1024", **_gemm(1024, 1024, 1024)),
        # odd sizes, both operands transposed, padded rows, update of C
        dict(name="sgemm_ragged_tt", **_gemm(1531, 1021, 777, op="TT", beta=0.5, pad=3)),
        # the largest: a square product that fills the chip for long
        dict(name="sgemm_8192", **_gemm(8192, 8192, 8192)),
        # the wide-range mode (three bf16 terms), weight-gradient layout, sizes that fit no tile
        dict(name="sgemm_tf32_nt", **_gemm(4000, 3000, 2000, mode="TF32TCEC", op="NT")),
        # outer-product-like: a large result of a short K
        dict(name="sgemm_short_k", **_gemm(16384, 16384, 256)),
        # a large matrix applied to a few vectors (decode of a batch, block Krylov)
        dict(name="sgemm_narrow", **_gemm(8192, 16, 8192, op="TN", data="normal")),
        # batched complex products of a circuit's tensor contraction
        dict(name="cgemm_batch_512", **_gemm(512, 512, 512, cplx=True, batch=64, data="unitary")),
        # many small real products of an odd size
        dict(name="sgemm_batch_100", **_gemm(100, 100, 100, batch=1000, data="normal")),
        # operands beyond fp16's range: maxima, power-of-two scaling and product
        dict(name="sgemm_scaling_4096", **_gemm(4096, 4096, 4096, mode="FP16TCEC_SCALING", data="spread")),
        # the library decides: statistics, decision on the device, product
        dict(name="cgemm_auto_1000", **_gemm(1000, 1000, 1000, mode="AUTO", cplx=True, data="unitary")),
        # one-qubit gate on a 27-qubit state vector: streaming
        dict(name="gate_27_qubits", **_gate(1 << 26)),
    ]


def _size(rng, lo, hi):
    """Spread over the logarithm; every other one a multiple of 32, the rest as they fall."""
    x = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    return max(lo, x // 32 * 32) if rng.random() < 0.5 and x >= 32 else max(lo, x)


def draw(rng):
    while True:
        kind = rng.choice(["real"] * 4 + ["complex"] * 2 + ["batch"] * 3 + ["narrow"] + ["decided"] * 2 + ["gate"])
        op = rng.choice(["NN", "TN", "NT", "TT"])
        beta = rng.choice([0.0, 0.0, 0.0, 1.0, 0.5])
        pad = rng.choice([0, 0, 0, 4, rng.randint(1, 33)])
        mode = rng.choice(["FP16TCEC"] * 4 + ["TF32TCEC"] * 2 + ["FP16TC", "TF32TC"])
        if kind == "gate":
            case = _gate(_size(rng, 1 << 12, 1 << 26), cplx=rng.random() < 0.7, wide=rng.random() < 0.3)
        elif kind == "batch":
            cplx = rng.random() < 0.4
            m, n, k = (_size(rng, 32, 768) for _ in range(3))
            if rng.random() < 0.5:
                n = k = m
            case = _gemm(m, n, k, mode, op, cplx, _size(rng, 4, 1024), beta, pad, "unitary" if cplx else "normal")
        elif kind == "narrow":
            few, many, k = rng.randint(1, 64), _size(rng, 1024, 16384), _size(rng, 256, 16384)
            m, n = (many, few) if rng.random() < 0.5 else (few, many)
            case = _gemm(m, n, k, mode, op, False, 1, beta, pad, "normal")
        else:
            cplx = kind == "complex" or (kind == "decided" and rng.random() < 0.3)
            m, n, k = (_size(rng, 64, 6144 if cplx else 10240) for _ in range(3))
            if rng.random() < 0.4:
                n = k = m
            if kind == "decided":
                mode = rng.choice(["AUTO", "FP16TCEC_SCALING"])
            data = "unitary" if cplx else ("spread" if mode == "FP16TCEC_SCALING" else rng.choice(["uniform", "normal"]))
            if cplx:
                op = op.replace("T", rng.choice("TC"))
            case = _gemm(m, n, k, mode, op, cplx, 1, beta, pad, data)
        w = work(case)
        if w["flops"] <= MOST_FLOPS and w["bytes"] <= MOST_BYTES:
            return case


def _stored(rows, cols, batch, pad, cplx, gen, data, dev, by_row=True):
    """A batch of column-major rows x cols matrices as a flat float tensor with leading dimension rows + pad, and
    that leading dimension.  `by_row`: which way the exponents of "spread" run."""
    ld = rows + pad
    shape = (batch, cols, ld) + ((2,) if cplx else ())
    if data == "uniform":
        x = torch.rand(shape, generator=gen, device=dev) * 2 - 1
    else:
        x = torch.randn(shape, generator=gen, device=dev)
    if data == "spread":
        # one integer exponent in [-30, 30] per row of A and per column of B: far outside fp16's range
        e = torch.randint(-30, 31, (batch, 1, ld) if by_row else (batch, cols, 1), generator=gen, device=dev)
        x = torch.ldexp(x, e[..., None] if cplx else e)
    return x.reshape(-1), ld


def _operands(case, seed):
    """The matrices of a case, made from the seed alone."""
    dev = torch.device("cuda")
    gen = torch.Generator(device=dev)
    gen.manual_seed(seed)
    s = {}
    cplx = case["cplx"]
    if case["kind"] == "gate":
        rows = case["rows"]
        s["x"] = torch.randn(2 * rows * (2 if cplx else 1), generator=gen, device=dev)
        g = torch.randn((2, 2, 2) if cplx else (2, 2), generator=gen, device=dev).cpu()
        q, _ = torch.linalg.qr(torch.view_as_complex(g) if cplx else g)
        s["u"] = (torch.view_as_real(q.contiguous()) if cplx else q).reshape(-1).to(dev)
        return s
    m, n, k, batch, pad = case["m"], case["n"], case["k"], case["batch"], case["pad"]
    op_a, op_b = case["op"]
    s["a"], s["lda"] = _stored(*((m, k) if op_a == "N" else (k, m)), batch, pad, cplx, gen, case["data"], dev,
                               by_row=op_a == "N")
    s["b"], s["ldb"] = _stored(*((k, n) if op_b == "N" else (n, k)), batch, pad, cplx, gen, case["data"], dev,
                               by_row=op_b != "N")
    s["ldc"] = m + pad
    if case["data"] == "unitary":  # entries of the size that a unitary's have
        s["a"] *= (2 * k) ** -0.5
        s["b"] *= (2 * k) ** -0.5
    c = torch.zeros(batch * n * s["ldc"] * (2 if cplx else 1), device=dev)
    if case["beta"]:
        c.normal_(generator=gen)
    s["c"] = c
    return s


def prepare(case, seed):
    s = _operands(case, seed)
    handle = cg.Handle()
    handle.set_stream(torch.cuda.current_stream())
    s["case"], s["handle"] = case, handle
    if case["kind"] == "gate":
        s["y"] = torch.zeros_like(s["x"])
    elif case["mode"] == "AUTO":
        # FP16TCEC while at most a tenth of the elements would lose their low half
        handle.set_exp_stats_params(0.0, 2.0 ** -15, 0.1)
    return s


def run(s):
    case, h = s["case"], s["handle"]
    cplx = case["cplx"]
    if case["kind"] == "gate":
        rows = case["rows"]
        if case["wide"]:
            st = h.gemm_2xNx2(cg.OP_N, cg.OP_N, rows, 1.0, s["u"], 2, s["x"], 2, 0.0, s["y"], 2, cplx=cplx)
        else:
            st = h.gemm_Mx2x2(cg.OP_N, cg.OP_N, rows, 1.0, s["x"], rows, s["u"], 2, 0.0, s["y"], rows, cplx=cplx)
        out = s["y"]
    else:
        m, n, k, batch = case["m"], case["n"], case["k"], case["batch"]
        op_a, op_b, mode = OPS[case["op"][0]], OPS[case["op"][1]], MODES[case["mode"]]
        a, b, c, lda, ldb, ldc, beta = s["a"], s["b"], s["c"], s["lda"], s["ldb"], s["ldc"], case["beta"]
        if mode in (cg.AUTO, cg.FP16TCEC_SCALING):
            st, _ = h.gemm_pipeline(op_a, op_b, m, n, k, 1.0, a, lda, b, ldb, beta, c, ldc, mode, cplx=cplx)
        elif batch > 1:
            st = h.gemm_strided_batch(op_a, op_b, m, n, k, 1.0, a, lda, a.numel() // batch // (2 if cplx else 1), b, ldb,
                                      b.numel() // batch // (2 if cplx else 1), beta, c, ldc, n * ldc, batch, mode,
                                      cplx=cplx)
        else:
            st = h.gemm(op_a, op_b, m, n, k, 1.0, a, lda, b, ldb, beta, c, ldc, mode, cplx=cplx)
        out = c
    if st != cg.STATUS_SUCCESS:
        raise RuntimeError(f"hipblasStatus {st}")
    return out


def work(case):
    es = 8 if case["cplx"] else 4
    if case["kind"] == "gate":
        return {"bytes": 4.0 * case["rows"] * es, "flops": 8.0 * case["rows"] * (4 if case["cplx"] else 1)}
    m, n, k, batch = case["m"], case["n"], case["k"], case["batch"]
    elements = m * k + k * n + m * n * (2 if case["beta"] else 1)
    return {"bytes": float(elements) * batch * es,
            "flops": 2.0 * m * n * k * batch * (4 if case["cplx"] else 1) * PRODUCTS[case["mode"]]}


def tolerance(case):
    # the products of a mode are the same in every correct implementation; what
    # differs is the order of FP32 sums (and, for the split modes, the last bit
    # of a split).  Measured against float64 products: 0.8 - 1.7e-7 for K up to
    # 1000, 5.8e-7 at K = 8192, the largest element 4 - 11 times that (77 times
    # for operands whose rows and columns differ in scale by 2^60); stated: about
    # four times as much.
    if case["kind"] == "gate":
        return {"rel": 4e-7, "max": 1e-5}
    rel = 2.0 ** -24 * (4.0 + 0.5 * math.sqrt(case["k"]))
    # (rows and columns of very different scale: single elements sit further from the root mean square)
    return {"rel": rel, "max": (64 if case["data"] == "spread" else 16) * rel}


def exact(case, seed):
    """What `run` returns, from products in 64 bits."""
    s = _operands(case, seed)
    cplx = case["cplx"]

    def parts(x):
        """Real and imaginary part (or the one part) of a stored operand, in 64 bits."""
        return [x.view(-1, 2)[:, i].double() for i in (0, 1)] if cplx else [x.double()]

    def product(p, q):
        if not cplx:
            return [p[0] @ q[0]]
        return [p[0] @ q[0] - p[1] @ q[1], p[0] @ q[1] + p[1] @ q[0]]

    def stored(xs):
        return torch.stack([x.reshape(-1) for x in xs], -1).reshape(-1)

    if case["kind"] == "gate":
        rows = case["rows"]
        x, u = parts(s["x"]), parts(s["u"])
        if case["wide"]:  # column-major 2 x rows, times the 2 x 2 matrix from the left
            return stored(product([p.view(rows, 2) for p in x], [p.view(2, 2) for p in u]))
        return stored(product([p.view(2, 2) for p in u], [p.view(2, rows) for p in x]))
    n, m, batch, ldc = case["n"], case["m"], case["batch"], s["ldc"]
    out = s["c"].double()
    per = out.numel() // batch
    a, b = s["a"].view(batch, -1), s["b"].view(batch, -1)

    def seen(x, op, ld, rows, cols):
        """op(X) transposed, rows x cols being op(X)'s own sizes."""
        if op == "N":
            xs = [p.view(cols, ld)[:, :rows] for p in parts(x)]
        else:
            xs = [p.view(rows, ld)[:, :cols].t() for p in parts(x)]
        return [xs[0], -xs[1]] if op == "C" else xs

    for i in range(batch):
        at = seen(a[i], case["op"][0], s["lda"], m, case["k"])
        bt = seen(b[i], case["op"][1], s["ldb"], case["k"], n)
        # row j of what a column-major matrix is in memory is its column j
        c = out[i * per:(i + 1) * per].view((n, ldc, 2) if cplx else (n, ldc, 1))[:, :m]
        c.copy_(torch.stack(product(bt, at), -1) + (case["beta"] * c if case["beta"] else 0))
    return out
