"""Performance cases of the GEMM library: what its users have it do, through its
public entry points, from one latency-bound call to a long prompt.

A case is one pass of `calls` GEMMs that share their activations (the
projections of one layer, or the same projection of consecutive layers), each
on weights and an output of its own.  Weights stay in HBM in the layout the
caller has them, and nothing but the library's calls is in a pass.  Kinds:

  sgemm      fp32, row-major; M <= 8 rows against streamed weights (decode,
             small batches), `beta` 1 where the layer adds into its output
  sgemm_tall fp32, many rows against a narrow B (a head, a 1x1 convolution)
  sgemm_ta   fp32, A stored K x M: the weight gradient of such a layer, a
             short output summed over all rows of a batch
  hook       fp32 inner product with bias through the oneDNN hook: weights
             N x K, as frameworks store them (encoder projections, MLPs)
  bf16       bf16 weights (K x N, or N x K with `nk`), fp32 accumulation and
             output: decode, short prompts, long prompts
  bf16_f32   the fp32-input bf16 entry (operands rounded to bf16 on the fly)
  s8         int8 x int8 -> int32, weights N x K
  s8_scale   the same with a per-column dequantization scale
  int8_f32   the fp32-input int8 entry (dynamic per-tensor quantization)
"""
import math
import os
import sys

import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "dnn-opt_amd", "python"))

import dnnopt_hip  # noqa: E402


def case(kind, M, N, K, calls=1, beta=0.0, nk=False):
    return {"kind": kind, "M": M, "N": N, "K": K, "calls": calls, "beta": beta, "nk": nk}


def listed():
    return [
        # The smallest call: two rows, a prime output width, one launch's latency.
        dict(case("sgemm", 2, 1009, 2048, beta=1.0), name="f32_two_rows"),
        # A small ragged batch through consecutive fp32 layers, added into their outputs: weights stream from HBM.
        dict(case("sgemm", 7, 11003, 2048, calls=4, beta=1.0), name="f32_ragged_batch"),
        # A narrow head over many rows.
        dict(case("sgemm_tall", 65536, 64, 256, calls=2), name="f32_tall_head"),
        # That head's weight gradient: 64 x 64 outputs over 262144 rows, A transposed.
        dict(case("sgemm_ta", 64, 64, 262144), name="f32_weight_grad"),
        # An encoder's MLP at 384 tokens: fp32 weights N x K, bias.
        dict(case("hook", 384, 3072, 768, calls=4, nk=True), name="f32_encoder_mlp"),
        # One decoded token through bf16 MLP projections.
        dict(case("bf16", 1, 11008, 4096, calls=4), name="bf16_decode"),
        # A short prompt (or a large decode batch) through the same weights.
        dict(case("bf16", 256, 11008, 4096, calls=4), name="bf16_short_prompt"),
        # A long prompt, weights N x K: the largest case.
        dict(case("bf16", 2048, 11008, 4096, nk=True), name="bf16_long_prompt"),
        # A prompt whose caller keeps everything in fp32 and asks for bf16 arithmetic.
        dict(case("bf16_f32", 512, 11008, 4096, calls=2), name="bf16_from_f32"),
        # int8 weights with a scale per output column, a medium batch.
        dict(case("s8_scale", 128, 4096, 4096, calls=8, nk=True), name="s8_scaled_batch"),
        # int8 weights, a long prompt, raw int32 sums.
        dict(case("s8", 1024, 11008, 4096, calls=2, nk=True), name="s8_prompt"),
        # fp32 tensors quantized per call.
        dict(case("int8_f32", 128, 4096, 4096, calls=4), name="int8_dynamic"),
    ]


# kind: ranges of M, N and K, and how many multiply-adds a pass of it may take
RANGES = {
    "sgemm": ((1, 8), (512, 11008), (1024, 4096), 2e9),
    "sgemm_tall": ((16384, 131072), (8, 64), (64, 256), 3e9),
    "sgemm_ta": ((33, 64), (33, 64), (32768, 262144), 3e9),
    "hook": ((16, 1024), (256, 4096), (256, 4096), 9e9),
    "bf16": ((1, 4096), (768, 11008), (768, 4096), 9e10),
    "bf16_f32": ((9, 1024), (768, 11008), (768, 4096), 4.6e10),
    "s8": ((5, 2048), (768, 11008), (768, 4096), 9e10),
    "s8_scale": ((1, 512), (768, 11008), (768, 4096), 9e10),
    "int8_f32": ((9, 512), (768, 4096), (768, 4096), 9e9),
}


def draw(rng):
    kind = rng.choice(sorted(RANGES))
    (m0, m1), (n0, n1), (k0, k1), most = RANGES[kind]

    def size(lo, hi, step):
        v = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
        # widths that divide evenly are the rule, odd ones the exception
        if rng.random() < 0.7:
            v = (v + step - 1) // step * step
        return max(lo, min(hi, v))

    M = size(m0, m1, 1 if m1 <= 64 else 16)
    N = size(n0, n1, 8 if n1 <= 64 else 64)
    K = size(k0, k1, 64)
    nk = kind in ("hook", "s8", "s8_scale") or (kind == "bf16" and rng.random() < 0.5)
    beta = 1.0 if kind in ("sgemm", "sgemm_tall", "bf16") and rng.random() < 0.3 else 0.0
    if kind in ("bf16", "s8", "s8_scale") and (K if nk else K | N) % 2:
        most = 2e10  # rows off 4-byte boundaries, as odd layers have them, in small and medium calls
    calls = rng.choice((1, 2, 4))
    while calls > 1 and float(M) * N * K * calls > most:
        calls //= 2
    while float(M) * N * K > most:
        M = max(m0, M // 2)
    return case(kind, M, N, K, calls, beta, nk)


def inputs(c, seed):
    """Activations, `calls` weights, outputs before the call, per-column vector (bias or scale)."""
    dev = torch.device("cuda:0")
    g = torch.Generator(device=dev).manual_seed(seed)
    M, N, K, kind = c["M"], c["N"], c["K"], c["kind"]
    a_shape = (K, M) if kind == "sgemm_ta" else (M, K)
    b_shape = (N, K) if c["nk"] else (K, N)

    def normal(shape, sigma):
        return torch.randn(shape, generator=g, device=dev).mul_(sigma)

    if kind in ("s8", "s8_scale"):
        A = torch.randint(-127, 128, a_shape, generator=g, device=dev, dtype=torch.int8)
        Bs = [torch.randint(-127, 128, b_shape, generator=g, device=dev, dtype=torch.int8) for _ in range(c["calls"])]
    else:
        A = normal(a_shape, 1.0)
        Bs = [normal(b_shape, 0.02) for _ in range(c["calls"])]
        if kind == "bf16":
            A, Bs = A.bfloat16(), [b.bfloat16() for b in Bs]
    out = torch.int32 if kind == "s8" else torch.float32
    if c["beta"]:
        Cs = [normal((M, N), 0.5) for _ in range(c["calls"])]
    else:
        Cs = [torch.zeros((M, N), dtype=out, device=dev) for _ in range(c["calls"])]
    vec = None
    if kind == "hook":
        vec = normal((N,), 0.1)
    elif kind == "s8_scale":
        vec = normal((N,), 1e-4).abs_().add_(1e-4)
    return A, Bs, Cs, vec


def prepare(c, seed):
    A, Bs, Cs, vec = inputs(c, seed)
    lib = dnnopt_hip.load()
    stream = torch.cuda.current_stream().cuda_stream
    return {"case": c, "lib": lib, "A": A, "Bs": Bs, "Cs": Cs, "vec": vec, "stream": stream}


def run(s):
    c, lib, A, Cs, vec, st = s["case"], s["lib"], s["A"], s["Cs"], s["vec"], s["stream"]
    kind, M, N, K, beta, nk = c["kind"], c["M"], c["N"], c["K"], c["beta"], c["nk"]
    ldb = K if nk else N
    for B, C in zip(s["Bs"], Cs):
        if kind in ("sgemm", "sgemm_tall"):
            lib.sgemm(M, N, K, 1.0, A, K, B, ldb, beta, C, N, transB=int(nk), stream=st)
        elif kind == "sgemm_ta":
            lib.sgemm(M, N, K, 1.0, A, M, B, ldb, beta, C, N, transA=1, stream=st)
        elif kind == "hook":
            # column-major: C^T (N x M) = W (N x K)^T-stored times x^T, bias per output feature
            lib.ext_sgemm("T", "N", N, M, K, 1.0, B, K, A, K, beta, C, N, bias=vec, stream=st)
        elif kind == "bf16":
            lib.gemm_bf16_ex(M, N, K, 1.0, A, K, B, ldb, beta, C, N, transB=int(nk), stream=st)
        elif kind == "bf16_f32":
            lib.gemm_bf16_f32in(M, N, K, 1.0, A, K, B, ldb, beta, C, N, stream=st)
        elif kind == "s8":
            lib.gemm_s8s8s32(M, N, K, A, K, B, K, C, N, stream=st)
        elif kind == "s8_scale":
            lib.gemm_s8s8f32_colscale(M, N, K, A, K, B, K, vec, C, N, stream=st)
        else:
            lib.gemm_int8_f32(M, N, K, 1.0, A, K, B, ldb, beta, C, N, stream=st)
    return Cs


def work(c):
    M, N, K, n, kind = c["M"], c["N"], c["K"], c["calls"], c["kind"]
    es = {"bf16": 2, "s8": 1, "s8_scale": 1}.get(kind, 4)
    vec = 4 * N if kind in ("hook", "s8_scale") else 0
    per_call = es * K * N + 4 * M * N * (2 if c["beta"] else 1)
    return {"bytes": float(es * M * K + vec + n * per_call), "flops": 2.0 * M * N * K * n}


def tolerance(c):
    if c["kind"] in ("s8", "s8_scale", "int8_f32"):
        # whole sums are exact, and every rounding after them is fixed by the interface
        return "exact"
    # fp32 sums of exact products in another order (bf16 operands multiply exactly in fp32)
    return {"rel": 4e-6, "max": 1e-4}


def exact(c, seed):
    A, Bs, Cs, vec = inputs(c, seed)
    kind = c["kind"]
    if kind == "bf16_f32":
        A, Bs = A.bfloat16(), [b.bfloat16() for b in Bs]
    scale = None
    if kind == "int8_f32":
        # the interface's quantizer (more than 8 rows): s = max|X| / 127 in fp32, q = rint(x * (1 / s))
        def quantize(x):
            s = x.abs().max() / 127.0
            return s, torch.clamp(torch.round(x * (1.0 / s)), -128, 127)

        sa, A = quantize(A)
        quantized = [quantize(b) for b in Bs]
        Bs, scale = [q for _, q in quantized], [sa.double() * sb.double() for sb, _ in quantized]
    a = A.double()
    a = a.t() if kind == "sgemm_ta" else a
    out = []
    for i, (B, C) in enumerate(zip(Bs, Cs)):
        b = B.double()
        v = a.contiguous() @ (b.t().contiguous() if c["nk"] else b)
        if c["beta"]:
            v += c["beta"] * C.double()
        if kind == "hook":
            v += vec.double()
        elif kind == "s8_scale":
            v *= vec.double()
        elif kind == "int8_f32":
            v *= scale[i]
        out.append(v)
    # whole sums are below 2^53, so they are exact here too
    return [v.to(torch.int32) for v in out] if kind == "s8" else out
