"""Performance cases of the EXL3 routed-expert path on one GPU: what a serving process calls, through the public entry
points, from one decoded token to a full 8192-token prefill chunk.

A case is a dict of plain values. `kind` selects the call:
  decode   exl3_grouped_runtime.moe_decode: one layer's routed experts for a small batch (fp32 out)
  prefill  exl3_grouped_runtime.grouped_prefill: one layer's routed experts for a prompt chunk
  router   exl3_grouped_runtime.grouped_prefill_from_logits: the router's top-k in front of the same
  linear   exl3_grouped.linear_exl3: a dense EXL3 projection (attention, shared expert)
  fat      exl3_grouped.fat_gemm_v2: one expert's GEMM over its gathered rows, the per-expert integration
  scatter  exl3_grouped.fat_gemm_v2_scatter: the same adding weighted rows into the layer output by token
Sizes are those of the repository's layer configurations (288 experts, hidden 4096, 768 or 1024 intermediate columns per
rank, top-8, 2 to 4 bits per weight) with token counts over the whole range between the smallest and the largest call.
"""
import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "glm53-exl3-prefill_amd"))

import exl3_grouped as ops  # noqa: E402
import exl3_grouped_runtime as rt  # noqa: E402

LIMIT = 10.0            # the layer's SwiGLU clamp
DECODE_CAP = 256        # rows a server sizes its decode workspace for
DTYPES = {"f16": torch.float16, "bf16": torch.bfloat16, "f32": torch.float32}


def _moe(name, kind, T, bits=4, I=768, routing="softmax", x="bf16", out="f32", E=288, H=4096, topk=8):
    return dict(name=name, kind=kind, T=T, E=E, H=H, I=I, topk=topk, bits=bits, routing=routing, x=x, out=out)


def _dense(name, kind, M, K, N, bits=4, out="f32"):
    return dict(name=name, kind=kind, M=M, K=K, N=N, bits=bits, out=out)


def listed():
    return [
        # one sequence being decoded: the latency a single user waits for, once per layer and token
        _moe("decode_1", "decode", 1),
        # a few sequences decoded together; fp16 activations
        _moe("decode_13", "decode", 13, x="f16"),
        # a full decode batch
        _moe("decode_96", "decode", 96),
        # a short prompt: every expert gets a handful of rows
        _moe("prefill_333", "prefill", 333, out="bf16"),
        # a 1024-token chunk with the router in front, balanced routing (about 28 rows per expert)
        _moe("router_1024", "router", 1024),
        # a ragged mid-size chunk, a few hot experts, the wider rank slice, 3 bits per weight
        _moe("prefill_2500_skewed_3b", "prefill", 2500, bits=3, I=1024, routing="skewed", out="bf16"),
        # the full chunk of a long prompt with popular experts: the benchmark's default workload
        _moe("prefill_8192_zipf", "prefill", 8192, routing="zipf", x="f16"),
        # a long chunk with 16 hot experts and 200 nearly idle ones, 2 bits per weight
        _moe("prefill_7168_thin_2b", "prefill", 7168, bits=2, routing="thin", out="bf16"),
        # a dense projection of a small decode batch (all that happens is reading its weights)
        _dense("linear_7", "linear", 7, 4096, 4096, out="f16"),
        # a dense projection of a prompt chunk
        _dense("linear_3000", "linear", 3000, 4096, 3072, out="f16"),
        # one expert's gate|up over a large batch, the per-expert integration
        _dense("fat_4096", "fat", 4096, 4096, 1536),
        # one expert's down projection for the rows routed to it, added into the chunk's output
        _dense("scatter_700", "scatter", 700, 768, 4096),
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(("decode", "decode", "prefill", "prefill", "prefill", "router", "linear", "fat", "scatter"))
    bits = rng.choice((4, 4, 3, 2))
    if kind in ("linear", "fat", "scatter"):
        K = 128 * rng.choice((6, 8, 16, 32))
        N = 128 * rng.choice((12, 16, 24, 32))
        M = _log_int(rng, 1 if kind == "linear" else 16, 4096)
        return dict(kind=kind, M=M, K=K, N=N, bits=bits, out=rng.choice(("f16", "f32")) if kind == "linear" else "f32")
    T = _log_int(rng, 1, 192) if kind == "decode" else _log_int(rng, 200, 6000)
    I = rng.choice((768, 768, 1024)) if T <= 4000 else 768
    c = _moe("", kind, T, bits=bits, I=I, routing=rng.choice(("softmax", "zipf", "thin", "skewed")),
             x=rng.choice(("bf16", "f16")), out=rng.choice(("f32", "bf16", "f16")) if kind == "prefill" else "f32")
    if kind == "router":
        c["routing"] = "softmax"
    del c["name"]
    return c


# ---------------------------------------------------------------------------------------------------- inputs
def _gen(seed, device="cpu"):
    return torch.Generator(device=device).manual_seed(int(seed))


def _routing(case, seed):
    """ids int64 [T, topk] (distinct per token) and fp32 weights summing to 1 per token, on the host."""
    T, E, k, kind = case["T"], case["E"], case["topk"], case["routing"]
    g = _gen(seed * 7 + 1)
    if kind in ("softmax", "zipf"):
        logits = torch.randn(T, E, generator=g)
        if kind == "zipf":                          # popularity of rank r ~ r^-1.1
            rank = torch.randperm(E, generator=g).double() + 1
            p = rank ** -1.1
            logits = logits + torch.log(p / p.sum()).float()
        v, ids = torch.topk(logits, k, dim=1)
        return ids, torch.softmax(v, dim=1)
    p = torch.full((E,), 0.0, dtype=torch.float64)
    perm = torch.randperm(E, generator=g)
    if kind == "thin":                              # 16 hot experts hold 60%, 200 get about 8 rows each
        rows = T * k
        hot, thin, warm = perm[:16], perm[16:216], perm[216:]
        thin_share = min(0.2, 200 * 8.0 / rows)
        p[hot], p[thin] = 0.6 / 16, thin_share / 200
        p[warm] = (0.4 - thin_share) / len(warm)
    else:                                           # skewed: 12 experts take 55% beside their uniform share
        p[:] = 0.45 / E
        p[perm[:12]] += 0.55 / 12
    u = torch.rand(T, E, generator=g, dtype=torch.float64).clamp_(1e-12, 1 - 1e-12)
    ids = torch.topk(torch.log(p) - torch.log(-torch.log(u)), k, dim=1).indices     # without replacement, ~ p
    w = torch.rand(T, k, generator=g) + 1e-3
    return ids, (w / w.sum(1, keepdim=True)).float()


def _words(shape, g):
    return torch.randint(-32768, 32768, shape, dtype=torch.int16, device="cuda", generator=g)


def _signs(shape, g):
    return (torch.randint(0, 2, shape, dtype=torch.int8, device="cuda", generator=g) * 2 - 1).to(torch.float16)


def _scales(shape, K, g):
    """Output scales: sign x U(0.5, 1.5) / sqrt(K), so that a projection of unit rows has unit rows."""
    u = torch.rand(shape, device="cuda", generator=g) + 0.5
    return (u * _signs(shape, g).float() / math.sqrt(K)).to(torch.float16)


class Layer:
    """The attributes the runtime reads from a routed-expert layer."""

    def __init__(self, case, seed):
        E, H, I, w = case["E"], case["H"], case["I"], 16 * case["bits"]
        g = _gen(seed * 7 + 2, "cuda")
        self.w13_trellis = _words((E, 2, H // 16, I // 16, w), g)
        self.w2_trellis = _words((E, I // 16, H // 16, w), g)
        self.w13_suh = _signs((E, 1, H), g).expand(E, 2, H).contiguous()
        self.w13_svh = _scales((E, 2, I), H, g)
        self.w2_suh = _signs((E, I), g)
        self.w2_svh = _scales((E, H), I, g)
        self._exl3_intermediate_local = I


def _inputs(case, seed):
    g = _gen(seed * 7 + 3, "cuda")
    s = {"case": case}
    if case["kind"] in ("decode", "prefill", "router"):
        T, H, E = case["T"], case["H"], case["E"]
        s["layer"] = Layer(case, seed)
        s["x"] = torch.randn(T, H, device="cuda", generator=g).to(DTYPES[case["x"]])
        if case["kind"] == "router":
            s["logits"] = torch.randn(T, E, device="cuda", generator=g).to(torch.bfloat16)
            s["bias"] = torch.randn(E, device="cuda", generator=g) * 0.05
        else:
            ids, w = _routing(case, seed)
            s["ids"], s["w"] = ids.cuda(), w.cuda()
        return s
    M, K, N = case["M"], case["K"], case["N"]
    s["x"] = torch.randn(M, K, device="cuda", generator=g).to(torch.float16)
    s["packed"] = _words((K // 16, N // 16, 16 * case["bits"]), g)
    s["svh"] = _scales((N,), K, g)
    if case["kind"] == "linear":
        s["suh"] = _signs((K,), g)
    if case["kind"] == "scatter":
        tokens = 4 * M
        s["tok"] = torch.randperm(tokens, device="cuda", generator=g)[:M].sort().values
        s["rw"] = torch.rand(M, device="cuda", generator=g).to(torch.float16)
    return s


def prepare(case, seed):
    s = _inputs(case, seed)
    kind = case["kind"]
    if kind == "decode":
        # a server sizes the decode workspace once, for its row cap
        rt.reserve_decode_workspace(torch.device("cuda", torch.cuda.current_device()), DECODE_CAP, 8, 288, 4096, 1024)
    elif kind == "linear":
        s["work"] = torch.empty(max(16, ops.linear_workspace_bytes(case["M"], case["K"])), dtype=torch.uint8,
                                device="cuda")
    elif kind == "fat":
        s["out"] = torch.empty(case["M"], case["N"], device="cuda")
    elif kind == "scatter":
        s["out"] = torch.empty(4 * case["M"], case["N"], device="cuda")
    return s


def run(s):
    c = s["case"]
    kind = c["kind"]
    if kind == "decode":
        return rt.moe_decode(s["x"], s["ids"], s["w"], s["layer"], LIMIT)
    if kind == "prefill":
        return rt.grouped_prefill(s["x"], s["ids"], s["w"], s["layer"], LIMIT,
                                  out_dtype=None if c["out"] == "f32" else DTYPES[c["out"]])
    if kind == "router":
        return rt.grouped_prefill_from_logits(s["x"], s["logits"], s["layer"], LIMIT, s["bias"], topk=c["topk"])
    if kind == "linear":
        return ops.linear_exl3(s["x"], s["packed"], s["suh"], s["svh"], K=c["bits"], out_dtype=DTYPES[c["out"]],
                               work=s["work"])
    if kind == "fat":
        ops.fat_gemm_v2(s["x"], s["packed"], s["out"], s["svh"], c["bits"], True, False)
        return s["out"]
    s["out"].zero_()                                # the chunk's output, which every expert adds into
    ops.fat_gemm_v2_scatter(s["x"], s["packed"], s["out"], s["svh"], s["tok"], s["rw"], c["bits"], True, False)
    return s["out"]


# ---------------------------------------------------------------------------------------------------- reference
def work(case):
    if case["kind"] in ("decode", "prefill", "router"):
        T, H, I, k = case["T"], case["H"], case["I"], case["topk"]
        if case["kind"] == "router":
            active = case["E"] * (1 - (1 - k / case["E"]) ** T)
        else:
            active = int(torch.unique(_routing(case, 0)[0]).numel())
        weights = active * (3 * H * I * case["bits"] / 8 + 2 * (2 * H + 3 * I))
        out = T * H * (4 if case["out"] == "f32" else 2)
        return {"bytes": weights + 2 * T * H + out + 12 * T * k, "flops": 6.0 * T * k * H * I}
    M, K, N = case["M"], case["K"], case["N"]
    out = M * N * (2 if case["out"] == "f16" else 4)
    if case["kind"] == "scatter":
        out = 4 * M * N * 4
    return {"bytes": K * N * case["bits"] / 8 + 2 * M * K + out, "flops": 2.0 * M * K * N}


def tolerance(case):
    # four times what the path measures against `exact`; another summation order moves it by far less
    if case["kind"] in ("fat", "scatter"):
        return {"rel": 2e-6}                        # exact fp16 operands, 32-bit sums: 2e-7 to 4e-7
    if case["kind"] == "linear":
        return {"rel": 1.2e-3}                      # the rotated rows in fp16, and the fp16 output: 2.9e-4
    return {"rel": 7.2e-3 if case["out"] == "bf16" else 2.6e-3}     # three fp16 roundings 5.7e-4; bf16 output 1.8e-3


def _code_table(device):
    """The 65536 code values: x = s * 0xCBAC1FED mod 2^32, masked and xored, its two fp16 halves added in fp16."""
    s = torch.arange(65536, dtype=torch.int64, device=device)
    y = ((s * 0xCBAC1FED) & 0x8FFF8FFF) ^ 0x3B603B60
    lo, hi = (y & 0xFFFF), (y >> 16) & 0xFFFF
    as_f16 = lambda v: torch.where(v >= 32768, v - 65536, v).to(torch.int16).view(torch.float16)  # noqa: E731
    return (as_f16(lo).float() + as_f16(hi).float()).to(torch.float16).double()


def _weights(packed, bits, table):
    """W' [16 tiles_k, 16 tiles_n] in float64 from trellis words [tiles_k, tiles_n, 16 bits]."""
    tk, tn, words = packed.shape
    dev = packed.device
    w = packed.to(torch.int64) & 0xFFFF
    p = torch.arange(256, device=dev)
    start = ((p + 1) * bits - 16) % (256 * bits)    # the first of the state's 16 stream bits
    a, sh = start // 16, start % 16
    two = w[..., a] | (w[..., (a + 1) % words] << 16)
    v = table[(two >> sh) & 0xFFFF]                 # [tk, tn, 256]
    c, j = p // 8, p % 8
    k = 2 * (c & 3) + (j & 1) + 8 * ((j >> 1) & 1)
    n = (c >> 2) + 8 * (j >> 2)
    out = torch.empty(tk, tn, 16, 16, dtype=torch.float64, device=dev)
    out[:, :, k, n] = v
    return out.permute(0, 2, 1, 3).reshape(tk * 16, tn * 16)


def _had(x):
    """Walsh-Hadamard over each 128-column block, orthonormal."""
    h = torch.ones(1, 1, dtype=torch.float64, device=x.device)
    for _ in range(7):
        h = torch.cat((torch.cat((h, h), 1), torch.cat((h, -h), 1)), 0)
    return (x.reshape(-1, 128) @ h / math.sqrt(128)).reshape(x.shape)


def _project(h, packed, svh, bits, table):
    return _had(h @ _weights(packed, bits, table)) * svh.double()


def exact(case, seed):
    s = _inputs(case, seed)
    bits, x = case["bits"], s["x"].double()
    table = _code_table(x.device)
    if case["kind"] == "linear":
        return _project(_had(x * s["suh"].double()), s["packed"], s["svh"], bits, table)
    if case["kind"] in ("fat", "scatter"):
        y = _project(x, s["packed"], s["svh"], bits, table)
        if case["kind"] == "fat":
            return y
        out = torch.zeros(4 * case["M"], case["N"], dtype=torch.float64, device=x.device)
        return out.index_add_(0, s["tok"], y * s["rw"].double()[:, None])
    if case["kind"] == "router":
        score = torch.sigmoid(s["logits"].double())
        ids = torch.topk(score + s["bias"].double(), case["topk"], dim=1).indices
        w = torch.gather(score, 1, ids)
        w = w / w.sum(1, keepdim=True) * 2.5
    else:
        ids, w = s["ids"], s["w"].double()
    L = s["layer"]
    out = torch.zeros(case["T"], case["H"], dtype=torch.float64, device=x.device)
    for e in torch.unique(ids).tolist():
        t, j = torch.nonzero(ids == e, as_tuple=True)
        h = _had(x[t] * L.w13_suh[e, 0].double())
        g = _project(h, L.w13_trellis[e, 0], L.w13_svh[e, 0], bits, table).clamp(max=LIMIT)
        u = _project(h, L.w13_trellis[e, 1], L.w13_svh[e, 1], bits, table).clamp(-LIMIT, LIMIT)
        a = _had(g * torch.sigmoid(g) * u * L.w2_suh[e].double())
        y = _project(a, L.w2_trellis[e], L.w2_svh[e], bits, table)
        out.index_add_(0, t, y * w[t, j][:, None])
    return out
