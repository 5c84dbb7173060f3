"""What a user of the framework has it do, as cases that can be timed.

A case names one call of the public API with its sizes and options; `prepare` makes what the
caller holds before it (operands, output, workspace, operands split once), `run` is the call.
Kinds:
  matmul    tcec.matmul_tn: C = A B^T of two contiguous row-major matrices, the result allocated
            by the call
  sgemm     tcec.sgemm: the BLAS-style product, any transposes, leading dimensions, alpha / beta
  strided   tcec.sgemm_strided_batched
  pointers  tcec.sgemm_batched on device arrays of matrix pointers, the convention of the
            reference's GEMM harness (test/tcec/batch_gemm.cu:433-443)
  packed    a weight matrix split once (tcec.pack, outside the call), then per call the pack of
            the other operand and tcec.gemm_packed
  api       tcec.api_gemm: the GEMM written against the header-only device API
  tiles     tcec.primitive_tiles: the fragment primitives over a stream of 16x16 tiles
"""
import math

import torch

from wmma_extension_amd import tcec

# matrix products issued per effective product, by policy
PRODUCTS = {"F16_EC": 3, "F16_NOEC": 1, "BF16X3_EC": 6, "BF16X2_EC": 3, "BF16_NOEC": 1}
TERMS = {"F16_EC": 2, "F16_NOEC": 1, "BF16X3_EC": 3, "BF16X2_EC": 2, "BF16_NOEC": 1}
# device-API operand type and error correction of each policy (tcec.api_gemm)
API_TYPE = {"F16_EC": (0, 1), "F16_NOEC": (0, 0), "BF16X3_EC": (2, 1), "BF16X2_EC": (1, 1), "BF16_NOEC": (1, 0)}


def _gemm(kind, m, n, k, policy="F16_EC", ta="T", tb="N", batch=1, alpha=1.0, beta=0.0, pad=0, rn=False,
          dist="normal", name=None):
    case = dict(kind=kind, m=m, n=n, k=k, policy=policy, ta=ta, tb=tb, batch=batch, alpha=alpha, beta=beta,
                pad=pad, rn=rn, dist=dist)
    if name is not None:
        case["name"] = name
    return case


def listed():
    return [
        # the smallest call: one 64^3 product, all latency (a preconditioner block, a small solve)
        _gemm("matmul", 64, 64, 64, dist="uniform", name="matmul_64"),
        # the ordinary single product, a few dozen microseconds
        _gemm("matmul", 1024, 1024, 1024, dist="uniform", name="matmul_1024"),
        # the product of the headline metric that the fp16 policy is used for
        _gemm("matmul", 4096, 4096, 4096, dist="uniform", name="matmul_4096"),
        # the largest: the full fp32 range through three bf16 terms
        _gemm("matmul", 16384, 16384, 16384, policy="BF16X3_EC", dist="exp", name="matmul_16384_bf16x3"),
        # row-major A B of a host program (column-major B^T A^T, no transposes), a few entries of odd
        # sizes, alpha and beta in use, fp32 range
        _gemm("strided", 777, 1333, 515, policy="BF16X3_EC", ta="N", tb="N", batch=7, alpha=0.5, beta=0.5,
              dist="normal", name="ragged_nn_7x777x1333x515_bf16x3"),
        # the gradient of a linear layer's weights: neither operand has k contiguous, added to what is there
        _gemm("sgemm", 1024, 3072, 4096, ta="N", tb="T", beta=1.0, dist="normal", name="grad_nt_1024x3072x4096"),
        # many small matrices at once
        _gemm("strided", 256, 256, 256, batch=1024, dist="normal", name="strided_1024x256"),
        # the reference harness's grid, 256 entries by pointer
        _gemm("pointers", 1024, 1024, 1024, batch=256, dist="uniform", name="pointers_256x1024"),
        # a K-heavy product: few outputs, long sums
        _gemm("sgemm", 1024, 1024, 262144, dist="normal", name="kheavy_1024x1024x262144"),
        # weights split once, activations of one batch per call
        _gemm("packed", 4096, 512, 4096, dist="normal", name="packed_4096x512x4096"),
        # a GEMM on the header-only device API
        _gemm("api", 4096, 4096, 4096, dist="uniform", name="api_4096"),
        # the fragment primitives over the benchmark's stream of tiles
        {"name": "tiles_1M", "kind": "tiles", "tiles": 1 << 20},
    ]


def _size(rng, lo, hi):
    """lo .. hi, even over the logarithm; half of them multiples of 32 (16, 8, .. below 32)."""
    v = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    if rng.random() < 0.5 and v >= 32:
        v = 32 * max(1, round(v / 32))
    return max(lo, min(hi, v))


def draw(rng):
    while True:
        kind = rng.choice(["matmul", "matmul", "sgemm", "sgemm", "sgemm", "strided", "strided", "strided",
                           "pointers", "pointers", "packed", "api", "tiles"])
        if kind == "tiles":
            return dict(kind="tiles", tiles=int(round(2 ** rng.uniform(10, 20))))
        policy = rng.choice(["F16_EC"] * 5 + ["BF16X3_EC"] * 3 + ["BF16X2_EC", "F16_NOEC", "BF16_NOEC"])
        batch = 1
        if kind == "api":
            m, n = 128 * rng.randint(2, 48), 128 * rng.randint(2, 48)
            k = 32 * _size(rng, 4, 256)
        elif kind in ("strided", "pointers"):
            batch = _size(rng, 2, 1024)
            m, n, k = _size(rng, 32, 2048), _size(rng, 32, 2048), _size(rng, 32, 16384)
        else:
            m, n, k = _size(rng, 32, 8192), _size(rng, 32, 8192), _size(rng, 32, 65536)
        elems = (m * k + k * n + 2 * m * n) * batch
        flops = 2.0 * m * n * k * batch
        # a state of at most about 2 GiB of operands; no costlier than the largest listed product
        if elems > 1 << 29 or flops > 4e12:
            continue
        ta = tb = None
        if kind in ("matmul", "pointers", "packed", "api"):
            ta, tb = "T", "N"
        else:
            ta, tb = rng.choice([("T", "N"), ("T", "N"), ("N", "N"), ("N", "T"), ("T", "T")])
        alpha, beta = rng.choice([(1.0, 0.0), (1.0, 0.0), (1.0, 1.0), (0.5, 0.5)])
        if kind == "matmul":
            alpha, beta = 1.0, 0.0
        pad = rng.choice([0, 0, 0, 4, 5]) if kind in ("sgemm", "strided") else 0
        rn = kind not in ("api", "packed") and policy in ("F16_EC", "BF16X3_EC") and rng.random() < 0.1
        dist = rng.choice(["uniform", "normal"] if policy.startswith("F16") else ["uniform", "normal", "exp"])
        return _gemm(kind, m, n, k, policy, ta, tb, batch, alpha, beta, pad, rn, dist)


def _values(case, shape, gen, dev):
    if case["dist"] == "normal":
        return torch.randn(shape, generator=gen, device=dev, dtype=torch.float32)
    v = torch.rand(shape, generator=gen, device=dev, dtype=torch.float32)
    if case["dist"] == "uniform":
        return v.mul_(2.0).sub_(1.0)
    # sign * [1, 2) * 2^e, e in -15 .. 15: the exponent range of fp32 in earnest
    e = torch.randint(-15, 16, shape, generator=gen, device=dev, dtype=torch.int8)
    s = torch.randint(0, 2, shape, generator=gen, device=dev, dtype=torch.int8)
    v.add_(1.0).mul_(1.0 - 2.0 * s)
    return torch.ldexp(v, e)


def prepare(case, seed):
    dev = torch.device("cuda:0")
    gen = torch.Generator(device=dev).manual_seed(seed)
    if case["kind"] == "tiles":
        return {"case": case, "tiles": torch.rand((case["tiles"], 256), generator=gen, device=dev).mul_(2.0).sub_(1.0)}
    m, n, k, batch, pad = case["m"], case["n"], case["k"], case["batch"], case["pad"]
    policy = tcec.Policy[case["policy"]]
    # column-major storage: the leading dimension is the inner one of the tensors below
    lda = (k if case["ta"] == "T" else m) + pad
    ldb = (k if case["tb"] == "N" else n) + pad
    ldc = m + pad
    A = _values(case, (batch, m if case["ta"] == "T" else k, lda), gen, dev)
    B = _values(case, (batch, n if case["tb"] == "N" else k, ldb), gen, dev)
    s = {"case": case, "policy": policy, "flags": tcec.FLAG_RN_MAIN if case["rn"] else 0, "A": A, "B": B,
         "lda": lda, "ldb": ldb, "ldc": ldc}
    if case["kind"] != "matmul":
        s["C"] = torch.randn((batch, n, ldc), generator=gen, device=dev, dtype=torch.float32)
    if case["kind"] == "packed":
        s["pa"] = torch.empty(tcec.pack_bytes(m, k, batch, policy), dtype=torch.uint8, device=dev)
        s["pb"] = torch.empty(tcec.pack_bytes(n, k, batch, policy), dtype=torch.uint8, device=dev)
        tcec.pack(policy, m, k, A, lda, 1, s["pa"])
        room = tcec.gemm_packed_workspace_bytes(policy, m, n, k, batch)
    elif case["kind"] != "api":
        room = tcec.workspace_bytes(m, n, k, batch, policy)
    else:
        room = 0
    s["ws"] = torch.empty(room, dtype=torch.uint8, device=dev) if room else None
    if case["kind"] == "pointers":
        for x in "ABC":
            s["p" + x] = torch.tensor([e.data_ptr() for e in s[x]], dtype=torch.int64, device=dev)
    return s


def run(s):
    c = s["case"]
    if c["kind"] == "tiles":
        return tcec.primitive_tiles(s["tiles"])
    m, n, k, batch, ta, tb, al, be = (c[x] for x in ("m", "n", "k", "batch", "ta", "tb", "alpha", "beta"))
    lda, ldb, ldc, policy, flags = s["lda"], s["ldb"], s["ldc"], s["policy"], s["flags"]
    if c["kind"] == "matmul":
        return tcec.matmul_tn(s["A"][0], s["B"][0], policy, flags, s["ws"])
    if c["kind"] == "sgemm":
        tcec.sgemm(ta, tb, m, n, k, al, s["A"], lda, s["B"], ldb, be, s["C"], ldc, policy, flags, s["ws"])
    elif c["kind"] == "strided":
        tcec.sgemm_strided_batched(ta, tb, m, n, k, al, s["A"], lda, s["A"].stride(0), s["B"], ldb,
                                   s["B"].stride(0), be, s["C"], ldc, s["C"].stride(0), batch, policy, flags,
                                   s["ws"])
    elif c["kind"] == "pointers":
        tcec.sgemm_batched(ta, tb, m, n, k, al, s["pA"], lda, s["pB"], ldb, be, s["pC"], ldc, batch, policy,
                           flags, s["ws"])
    elif c["kind"] == "packed":
        tcec.pack(policy, n, k, s["B"], ldb, 1, s["pb"])
        tcec.gemm_packed(policy, m, n, k, al, s["pa"], s["pb"], be, s["C"], ldc, workspace=s["ws"])
    else:
        type_, ec = API_TYPE[c["policy"]]
        tcec.api_gemm(type_, ec, m, n, k, al, s["A"], lda, s["B"], ldb, be, s["C"], ldc)
    return s["C"]


def work(case):
    """Operands and C once (C twice when beta reads it); the matrix products the policy is made of."""
    if case["kind"] == "tiles":
        # a tile in; four fragments of 64 lanes x 4 halves, the accumulator and the vectors out
        return {"bytes": case["tiles"] * (1024 + 4 * 512 + 1024 + 128), "flops": 0}
    m, n, k, batch = case["m"], case["n"], case["k"], case["batch"]
    a_bytes = 2 * TERMS[case["policy"]] if case["kind"] == "packed" else 4
    c_bytes = 8 if case["beta"] else 4
    return {"bytes": batch * (a_bytes * m * k + 4 * k * n + c_bytes * m * n),
            "flops": 2.0 * m * n * k * batch * PRODUCTS[case["policy"]]}


def tolerance(case):
    if case["kind"] == "tiles":
        return "exact"
    # fp32 sums. Against the same product in 64 bits (operands rounded as the policy rounds them) the
    # library is off by 6e-8 .. 1.3e-7 for short sums and up to 6.5e-9 sqrt(k) for long ones (4096:
    # 4.1e-7, 16384: 8.1e-7), 1.2e-6 for the 262144-long one; no value by more than 8 times the
    # relative error.  Four times that.
    rel = min(5e-6, max(5e-7, 2.6e-8 * math.sqrt(case["k"])))
    return {"rel": rel, "max": 8 * rel}
