"""Timed cases of the library: what a program that calls it runs, through the
package's public entry points (7_amd/ops.py).

Four kinds of work, each over the sizes, types and options a caller uses:

* ``gemm`` / ``auto``: C = A . B^T (``gemm``: the fixed entry point,
  ``gemm_auto``: the shape-driven one with the workspace a program keeps),
  f16 or bf16 in, f32 / f16 / bf16 out, row- or column-major C;
* ``mxfp4``: the scaled 4-bit GEMM, canonical or AITER input layout;
* ``fwd`` / ``train`` / ``mxfp8``: flash attention -- the forward alone (with
  or without a causal mask, grouped-query heads, the fixed-max mode), the
  forward and backward of a training step, and the block-scaled FP8 forward
  with the quantisation of its inputs;
* ``f32``: the single-tile attention with f32 output.

``listed()`` names the workloads; ``draw()`` gives other sizes and options of
the same ranges.  Inputs follow the distributions of the library's benchmark:
f16 GEMM operands uniform in [-1, 1), bf16 ones N(0, 1) / sqrt(K), attention
inputs N(0, 1) (uniform within the declared bound in the fixed-max mode),
random fp4 codes with scales around one.
"""

import importlib
import math

import torch

wave = importlib.import_module("7_amd")

DT = {"f16": torch.float16, "bf16": torch.bfloat16, "f32": torch.float32}
D = 128  # head dimension of the flash-attention kernels


def listed():
    return [
        # The smallest call: one 32 x 32 tile of f32 output.  Launch and host
        # latency.
        dict(name="gemm_f16_32x32x64", kind="gemm", M=32, N=32, K=64, dt="f16", out="f32",
             layout="row"),
        # An ordinary square product, e.g. a projection of a small model.
        dict(name="gemm_f16_1024", kind="gemm", M=1024, N=1024, K=1024, dt="f16", out="f16",
             layout="row"),
        # Ragged M and K: a projection over a batch of tokens whose count is no
        # multiple of anything.
        dict(name="gemm_bf16_4000x4096x4100", kind="gemm", M=4000, N=4096, K=4100, dt="bf16",
             out="bf16", layout="row"),
        # The largest product (the library's headline benchmark).
        dict(name="gemm_f16_8192", kind="gemm", M=8192, N=8192, K=8192, dt="f16", out="f16",
             layout="row"),
        # Few rows against a large weight matrix: a decoding step of a batch,
        # bound by reading the weights.
        dict(name="auto_bf16_128x8192x8192", kind="auto", M=128, N=8192, K=8192, dt="bf16",
             out="bf16", layout="row"),
        # A small output with a long sum: the reference's split Stream-K shape
        # (column-major C, as it stores it).
        dict(name="auto_f16_2048x2048x8192", kind="auto", M=2048, N=2048, K=8192, dt="f16",
             out="f16", layout="col"),
        # 4-bit weights and activations.
        dict(name="mxfp4_4096x4096x8192", kind="mxfp4", M=4096, N=4096, K=8192, out="f16",
             layout="col", aiter=False),
        # Attention over long sequences (the library's headline benchmark).
        dict(name="fwd_f16_b4_h32_s4096", kind="fwd", B=4, Hq=32, Hkv=32, S=4096, dt="f16",
             causal=False, qk_max=0.0),
        # Prefill of one prompt of odd length, grouped-query heads, causal.
        dict(name="fwd_bf16_gqa_s1000", kind="fwd", B=1, Hq=32, Hkv=8, S=1000, dt="bf16",
             causal=True, qk_max=0.0),
        # The attention of a training step: forward with its row statistics,
        # then the backward.
        dict(name="train_bf16_gqa_s2048", kind="train", B=2, Hq=16, Hkv=4, S=2048, dt="bf16",
             causal=True),
        # Attention on FP8 inputs: quantise q, k and v, then the forward.
        dict(name="mxfp8_bf16_gqa_s2048", kind="mxfp8", B=2, Hq=32, Hkv=8, S=2048, dt="bf16",
             causal=False),
        # One tile of queries against a context, f32 output.
        dict(name="f32_64x1024x64", kind="f32", M=64, S=1024, D=64),
    ]


def _log(rng, lo, hi, steps):
    """A whole number spread over [lo, hi] by its logarithm, rounded to a
    multiple of one of `steps` (picked at random; 1 leaves odd numbers)."""
    n = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    g = rng.choice(steps)
    return max(g if g >= lo else lo, min(hi, (n + g // 2) // g * g))


def draw(rng):
    kind = rng.choice(["gemm", "gemm", "auto", "auto", "mxfp4", "fwd", "fwd", "train", "mxfp8",
                       "f32"])
    dt = rng.choice(["f16", "bf16"])
    if kind == "gemm":
        # Whole tiles, ragged ones, and sizes without any alignment; at most a
        # quarter of the largest listed product's work, far less without
        # alignment (K off 4 elements reads element by element).
        while True:
            M = _log(rng, 32, 8192, [64, 256, 1])
            N = _log(rng, 32, 8192, [64, 256, 8, 1])
            K = _log(rng, 32, 8192, [64, 64, 8, 4, 1])
            if M * N * K <= (2 ** 37 if K % 4 == 0 else 2 ** 33):
                break
        return dict(kind=kind, M=M, N=N, K=K, dt=dt, out=rng.choice([dt, dt, "f32"]),
                    layout=rng.choice(["row", "row", "col"]))
    if kind == "auto":
        if rng.random() < 0.6:  # a few rows: decoding steps of 1 to 128 sequences
            M = _log(rng, 1, 128, [1])
            N, K = (_log(rng, 1024, 16384, [64, 256, 8]) for _ in range(2))
            K = max(64, K // 64 * 64)
        else:  # small outputs, long sums
            M, N = (_log(rng, 129, 2048, [64, 256, 1]) for _ in range(2))
            K = _log(rng, 1024, 16384, [64, 64, 8])
        return dict(kind=kind, M=M, N=N, K=K, dt=dt, out=dt,
                    layout="row" if N % 4 == 0 and rng.random() < 0.7 else "col")
    if kind == "mxfp4":
        M, N = (_log(rng, 256, 4096, [256]) for _ in range(2))
        return dict(kind=kind, M=M, N=N, K=_log(rng, 256, 16384, [128, 256]),
                    out=rng.choice(["f16", "bf16", "f32"]), layout=rng.choice(["row", "col"]),
                    aiter=rng.random() < 0.3)
    if kind == "f32":
        return dict(kind=kind, M=_log(rng, 1, 128, [16, 1]), S=_log(rng, 16, 4096, [64, 1]),
                    D=_log(rng, 16, 128, [32, 8, 1]))
    Hq = rng.choice([1, 4, 8, 16, 32, 64])
    Hkv = max(1, Hq // rng.choice([1, 1, 4, 8]))
    B = rng.choice([1, 1, 2, 4, 8])
    causal = rng.random() < 0.5
    if kind == "train":  # the backward takes whole 64-row blocks
        S = _log(rng, 64, 4096, [64, 128])
        while B * Hq * S * S > 2 ** 28:
            S = S // 128 * 64
        return dict(kind=kind, B=B, Hq=Hq, Hkv=Hkv, S=max(64, S), dt=dt, causal=causal)
    S = _log(rng, 16, 8192, [64, 1])
    while B * Hq * S * S > 2 ** 30:
        S //= 2
    case = dict(kind=kind, B=B, Hq=Hq, Hkv=Hkv, S=S, dt=dt, causal=causal)
    if kind == "fwd":
        bounded = rng.random() < 0.2  # inputs with a known bound: the fixed-max mode
        case["qk_max"] = 0.0 if not bounded else 1.0 if dt == "bf16" else 0.5
    return case


# ------------------------------------------------------------------ inputs

def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _rand(case, seed):
    g = torch.Generator(device=_device())
    g.manual_seed(seed)

    def normal(*shape, scale=1.0):
        return torch.randn(shape, generator=g, device=g.device, dtype=torch.float32) * scale

    def uniform(*shape, bound=1.0):
        return (torch.rand(shape, generator=g, device=g.device, dtype=torch.float32) * 2 - 1) * bound

    def whole(lo, hi, *shape):
        return torch.randint(lo, hi, shape, generator=g, device=g.device, dtype=torch.int32)

    return normal, uniform, whole


def _inputs(case, seed):
    normal, uniform, whole = _rand(case, seed)
    kind = case["kind"]
    if kind in ("gemm", "auto"):
        M, N, K, dt = case["M"], case["N"], case["K"], DT[case["dt"]]
        if case["dt"] == "f16":
            return uniform(M, K).to(dt), uniform(N, K).to(dt)
        return (normal(M, K, scale=K ** -0.5).to(dt), normal(N, K, scale=K ** -0.5).to(dt))
    if kind == "mxfp4":
        M, N, K = case["M"], case["N"], case["K"]
        a, b = whole(0, 256, M, K // 2).to(torch.uint8), whole(0, 256, N, K // 2).to(torch.uint8)
        sa, sb = (whole(123, 130, K // 32, n).to(torch.uint8) for n in (M, N))
        return a, b, sa, sb
    if kind == "f32":
        M, S, d = case["M"], case["S"], case["D"]
        q = normal(M, d, scale=math.log2(math.e) / math.sqrt(d)).to(torch.float16)
        return q, normal(S, d).to(torch.float16), normal(S, d).to(torch.float16)
    B, Hq, Hkv, S, dt = case["B"], case["Hq"], case["Hkv"], case["S"], DT[case["dt"]]
    if case.get("qk_max", 0.0) > 0.0:
        q = uniform(B, Hq, S, D, bound=case["qk_max"]).to(dt)
        k = uniform(B, Hkv, S, D, bound=case["qk_max"]).to(dt)
    else:
        q, k = normal(B, Hq, S, D).to(dt), normal(B, Hkv, S, D).to(dt)
    v = normal(B, Hkv, S, D).to(dt)
    return (q, k, v, normal(B, Hq, S, D).to(dt)) if kind == "train" else (q, k, v)


def _aiter_b(b):
    """[N, K/2] bytes in the AITER preshuffled order: 16-row blocks of
    [chunk of 32 bytes][half][row][16 bytes]."""
    N, KB = b.shape
    return b.view(N // 16, 16, KB // 32, 2, 16).permute(0, 2, 3, 1, 4).contiguous().view(N, KB)


def _aiter_scale(s):
    """[K/32, rows] scales as the AITER 256-byte blocks of 32 rows x 8 groups
    (groups padded to 8)."""
    G, R = s.shape
    G8 = (G + 7) // 8
    s = torch.nn.functional.pad(s, (0, 0, 0, G8 * 8 - G))
    return s.view(G8, 2, 4, R // 32, 2, 16).permute(3, 0, 2, 5, 1, 4).contiguous().view(-1)


def prepare(case, seed):
    kind = case["kind"]
    x = _inputs(case, seed)
    state = dict(case=case, x=x)
    if kind == "auto":
        need = wave.gemm_auto_workspace_bytes(case["M"], case["N"], case["K"])
        state["ws"] = torch.empty(need, dtype=torch.uint8, device=x[0].device) if need else None
    elif kind == "mxfp4" and case["aiter"]:
        a, b, sa, sb = x
        state["x"] = (a, _aiter_b(b), _aiter_scale(sa), _aiter_scale(sb))
    return state


def run(state):
    case, x = state["case"], state["x"]
    kind = case["kind"]
    if kind == "gemm":
        return wave.gemm(*x, out_dtype=case["out"], layout=case["layout"])
    if kind == "auto":
        return wave.gemm_auto(*x, out_dtype=case["out"], layout=case["layout"],
                              workspace=state["ws"])
    if kind == "mxfp4":
        return wave.gemm_mxfp4(*x, out_dtype=case["out"], layout=case["layout"],
                               input_layout="aiter" if case["aiter"] else "canonical")
    if kind == "f32":
        return wave.flash_attention_f32(*x)
    if kind == "fwd":
        return wave.flash_attention(*x, causal=case["causal"],
                                    qk_max_abs=case["qk_max"] or None)
    if kind == "train":
        q, k, v, do = x
        o, lse = wave.flash_attention_lse(q, k, v, causal=case["causal"])
        dq, dk, dv = wave.flash_attention_bwd(q, k, v, o, do, lse, causal=case["causal"])
        return dict(o=o, lse=lse, dq=dq, dk=dk, dv=dv)
    q, k, v = x
    (qe, qs), (ke, ks) = wave.mxfp8_quantize(q), wave.mxfp8_quantize(k)
    ve, vs = wave.mxfp8_quantize(v, dim=2)
    o = wave.flash_attention_mxfp8(qe, qs, ke, ks, ve, vs, causal=case["causal"],
                                   out_dtype=case["dt"])
    return dict(o=o, q=qe, q_scale=qs, k=ke, k_scale=ks, v=ve, v_scale=vs)


def work(case):
    kind = case["kind"]
    if kind in ("gemm", "auto"):
        M, N, K = case["M"], case["N"], case["K"]
        return dict(bytes=2 * K * (M + N) + M * N * (4 if case["out"] == "f32" else 2),
                    flops=2.0 * M * N * K)
    if kind == "mxfp4":
        M, N, K = case["M"], case["N"], case["K"]
        return dict(bytes=(K // 2 + K // 32) * (M + N) + M * N * (4 if case["out"] == "f32" else 2),
                    flops=2.0 * M * N * K)
    if kind == "f32":
        M, S, d = case["M"], case["S"], case["D"]
        return dict(bytes=2 * d * (M + 2 * S) + 4 * M * d, flops=4.0 * M * S * d)
    B, Hq, Hkv, S = case["B"], case["Hq"], case["Hkv"], case["S"]
    pairs = B * Hq * (S * (S + 1) / 2 if case["causal"] else S * S)  # (query, key) pairs
    qn, kn = B * Hq * S * D, B * Hkv * S * D
    if kind == "fwd":
        return dict(bytes=2 * (2 * qn + 2 * kn), flops=4.0 * D * pairs)
    if kind == "train":  # forward (q, k, v -> o, lse), backward (+ do -> dq, dk, dv)
        return dict(bytes=2 * (4 * qn + 4 * kn) + 4 * B * Hq * S, flops=14.0 * D * pairs)
    # q, k, v in; their bytes and scales and o out.
    return dict(bytes=2 * (2 * qn + 2 * kn) + (qn + 2 * kn) * 33 // 32, flops=4.0 * D * pairs)


def tolerance(case):
    """About four times the library's own distance from exact() (relative
    2-norm / largest), measured over the listed cases and thirty drawn ones:
    GEMM 3e-7 (f32 C, K = 2000; it grows with K), 2.1e-4 / 4.9e-4 (f16 C),
    1.7e-3 / 3.9e-3 (bf16 C); attention 2.9e-4 / 1.5e-3 (f16), 2.3e-3 / 6.1e-2
    (bf16, causal: the first rows' few terms cancel), its gradients 2.5e-3 /
    8.2e-2 (bf16); f32 attention 1.9e-4 / 8.7e-4 (f16 probabilities); FP8
    attention 2.6e-2 / 0.56 (probabilities in e4m3)."""
    kind = case["kind"]
    if kind in ("gemm", "auto", "mxfp4"):
        return {"f32": dict(rel=4e-6, max=2e-5), "f16": dict(rel=8e-4, max=2e-3),
                "bf16": dict(rel=7e-3, max=1.6e-2)}[case["out"]]
    if kind == "f32":
        return dict(rel=8e-4, max=4e-3)
    if kind == "mxfp8":
        return dict(rel=0.03, max=0.9)
    if case["dt"] == "f16":
        return dict(rel=1.3e-3, max=4e-2)
    return dict(rel=1e-2, max=0.3)


# ------------------------------------------------- the same results in 64 bits

_FP4 = (0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0, -0.0, -0.5, -1.0, -1.5, -2.0, -3.0, -4.0, -6.0)


def _fp4_decode(x, s):
    """[rows, K/2] codes and [K/32, rows] scales -> [rows, K] float64."""
    t = torch.tensor(_FP4, dtype=torch.float64, device=x.device)
    v = torch.stack((t[(x & 15).long()], t[(x >> 4).long()]), dim=-1).view(x.shape[0], -1)
    e = torch.exp2(s.double() - 127).t().repeat_interleave(32, dim=1)
    return v * e


def _mx8_decode(x, dim):
    """float64 values of the MX-FP8 encoding of x (blocks of 32 along `dim`,
    scale 2^(floor(log2 amax) - 8), elements rounded to e4m3, saturated)."""
    xs = x.double().movedim(dim, -1)
    n = xs.shape[-1]
    nb = -(-n // 32)
    b = torch.nn.functional.pad(xs, (0, nb * 32 - n)).reshape(*xs.shape[:-1], nb, 32)
    amax = b.abs().amax(dim=-1, keepdim=True)
    e = torch.where(amax > 0, torch.frexp(amax).exponent - 1.0 - 8.0, -127.0).clamp(-127, 127)
    scale = torch.exp2(e.double())
    q = (b / scale).clamp(-448.0, 448.0).float().to(torch.float8_e4m3fn).double() * scale
    return q.reshape(*xs.shape[:-1], nb * 32)[..., :n].movedim(-1, dim).contiguous()


def _attention(q, k, v, causal, do=None):
    """One head in float64: o, lse and, given do, dq, dk, dv."""
    scale = 1.0 / math.sqrt(D)
    s = (q @ k.t().contiguous()) * scale
    if causal:
        n = s.shape[0]
        s.masked_fill_(torch.ones(n, n, dtype=torch.bool, device=s.device).triu_(1), -math.inf)
    lse = torch.logsumexp(s, dim=1)
    p = s.sub_(lse[:, None]).exp_()
    o = p @ v
    if do is None:
        return o, lse
    dv = p.t().contiguous() @ do
    dp = do @ v.t().contiguous()
    ds = p.mul_(dp.sub_((do * o).sum(1, keepdim=True))).mul_(scale)
    return o, lse, ds @ k, ds.t().contiguous() @ q, dv


def exact(case, seed):
    x = _inputs(case, seed)
    kind = case["kind"]
    if kind in ("gemm", "auto", "mxfp4"):
        if kind == "mxfp4":
            a, b = _fp4_decode(x[0], x[2]), _fp4_decode(x[1], x[3])
        else:
            a, b = x[0].double(), x[1].double()
        return a @ b.t().contiguous() if case["layout"] == "row" else b @ a.t().contiguous()
    if kind == "f32":
        q, k, v = (t.double() for t in x)
        return torch.softmax((q @ k.t().contiguous()) * math.log(2.0), dim=1) @ v
    if kind == "mxfp8":
        x = (_mx8_decode(x[0], 3), _mx8_decode(x[1], 3), _mx8_decode(x[2], 2))
    q, k, v = (t.double() for t in x[:3])
    B, Hq, S, _ = q.shape
    group = Hq // k.shape[1]
    o = torch.empty_like(q)
    lse = torch.empty((B, Hq, S), dtype=torch.float64, device=q.device)
    dq, dk, dv = torch.empty_like(q), torch.zeros_like(k), torch.zeros_like(v)
    for b in range(B):
        for h in range(Hq):
            j = h // group
            if kind != "train":
                o[b, h], lse[b, h] = _attention(q[b, h], k[b, j], v[b, j], case["causal"])
                continue
            o[b, h], lse[b, h], dq[b, h], dkh, dvh = _attention(
                q[b, h], k[b, j], v[b, j], case["causal"], x[3][b, h].double())
            dk[b, j] += dkh
            dv[b, j] += dvh
    if kind == "fwd":
        return o
    if kind == "train":
        return dict(o=o, lse=lse, dq=dq, dk=dk, dv=dv)
    return dict(o=o, q=None, q_scale=None, k=None, k_scale=None, v=None, v_scale=None)
