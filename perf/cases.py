"""Performance cases: the work that a training or serving program has this framework do,
through its public entry points, over the sizes, types and options that it takes in earnest.

Kinds of case:
  linear          kernels.FP8Linear, forward and backward: y, dx, dw
  linear_infer    kernels.FP8Linear with its weight cache, forward only
  experts         moe.routed_experts, forward and backward: out, counts, dx, dw12, dw3, dscores
  experts_infer   moe.routed_experts with the weight cache, forward only
  indexer         kernels.indexer_scores_fp8, with the weights' gradient where "train"
  matmul          quantize_fp8_rowwise, quantize_fp8_blockwise and fp8_matmul_dsv3 on the
                  transposed weight codes: the calls of a program written for those functions
  grouped_f16     kernels.moe_grouped_gemm, the unquantized grouped product of the experts
  quantize        the two quantizers by themselves: codes and scales
"""
import math

import torch

from cinnamon_amd import kernels, layers, moe

BF16, F16, F32 = torch.bfloat16, torch.float16, torch.float32
_DT = {"bf16": BF16, "fp16": F16, "fp32": F32}


def listed():
    return [
        # the training step's dense projection at the headline size (config 2 and its backward)
        {"name": "linear_train_proj", "kind": "linear", "M": 8192, "K": 7168, "N": 2048, "x": "bf16", "w": "bf16",
         "round_scale": False},
        # a shared expert's w1 in the MTP block of the small training model (config 5): 16 x 1023
        # rows, fp32 master weights, power-of-two activation scales
        {"name": "linear_train_mtp", "kind": "linear", "M": 16368, "K": 1024, "N": 4096, "x": "bf16", "w": "fp32",
         "round_scale": True},
        # a small layer of a small batch (config 1): launches count
        {"name": "linear_train_small", "kind": "linear", "M": 2048, "K": 512, "N": 1024, "x": "bf16", "w": "bf16",
         "round_scale": False},
        # a generation step of 16 sequences through the same projection, weights quantized once
        {"name": "linear_decode", "kind": "linear_infer", "M": 16, "K": 7168, "N": 2048, "x": "bf16", "w": "bf16",
         "round_scale": False},
        # the large routed layer (config 3): 131072 ragged routed rows, the largest call there is
        {"name": "experts_train_large", "kind": "experts", "T": 16384, "D": 7168, "H": 2048, "E": 32, "k": 8,
         "x": "bf16"},
        # the routed layer of the small training model (config 5), batch 16 x 1024
        {"name": "experts_train", "kind": "experts", "T": 16384, "D": 1024, "H": 1024, "E": 16, "k": 2, "x": "bf16"},
        # a generation step of 64 sequences through the large routed layer
        {"name": "experts_decode", "kind": "experts_infer", "T": 64, "D": 7168, "H": 2048, "E": 32, "k": 8, "x": "bf16"},
        # the attention indexer in training (config 5): scores and the weights' gradient
        {"name": "indexer_train", "kind": "indexer", "B": 16, "L": 1024, "S": 1024, "H": 4, "d": 128, "x": "bf16",
         "train": True},
        # more and narrower heads, a ragged chunk of new tokens against a longer ragged context
        {"name": "indexer_prefill", "kind": "indexer", "B": 2, "L": 777, "S": 4100, "H": 8, "d": 64, "x": "bf16",
         "train": False},
        # a program that calls the quantizers and the product itself, at sizes no tile divides
        {"name": "matmul_ragged", "kind": "matmul", "M": 1000, "K": 4000, "N": 1500, "x": "bf16", "w": "bf16",
         "round_scale": False},
        # the unquantized routed layer's first product at the small training model's sizes
        {"name": "experts_f16", "kind": "grouped_f16", "T": 32768, "K": 1024, "N": 2048, "E": 16, "x": "bf16", "w": "fp32"},
        # the quantizers alone at the headline size
        {"name": "quantize", "kind": "quantize", "M": 8192, "K": 7168, "N": 2048, "x": "bf16", "w": "bf16",
         "round_scale": False},
    ]


# ---------------------------------------------------------------------------
# Drawn cases
# ---------------------------------------------------------------------------
def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _dim(rng, lo, hi):
    """A layer width: mostly whole 128s, some multiples of 16, a few odd."""
    n = _log(rng, lo, hi)
    step = rng.choice([128, 128, 128, 128, 16, 1])
    return max(lo, n // step * step)


def draw(rng):
    kind = rng.choice(["linear", "linear", "linear_infer", "experts", "experts_infer", "indexer", "matmul",
                       "grouped_f16", "quantize"])
    x = rng.choice(["bf16", "bf16", "bf16", "fp16", "fp32"])
    w = rng.choice(["fp32", "bf16"])
    rs = rng.random() < 0.3
    if kind in ("linear", "matmul", "quantize"):
        return {"kind": kind, "M": _log(rng, 64, 16384), "K": _dim(rng, 128, 7168), "N": _dim(rng, 128, 4096), "x": x,
                "w": w, "round_scale": rs}
    if kind == "linear_infer":
        return {"kind": kind, "M": _log(rng, 1, 256), "K": _dim(rng, 128, 7168), "N": _dim(rng, 128, 7168), "x": x, "w": w,
                "round_scale": rs}
    if kind in ("experts", "experts_infer"):
        E = rng.choice([4, 8, 16, 32, 64])
        return {"kind": kind, "T": _log(rng, 256, 16384) if kind == "experts" else _log(rng, 1, 256),
                "D": 128 * _log(rng, 2, 56 if E <= 32 else 28), "H": 128 * _log(rng, 2, 16), "E": E,
                "k": rng.choice([1, 2, 4, 8] if E >= 8 else [1, 2]), "x": x}
    if kind == "indexer":
        train = rng.random() < 0.5
        B, L = rng.choice([(_log(rng, 1, 16), _log(rng, 64, 1024)), (1, _log(rng, 512, 4096)), (_log(rng, 1, 64), 1)])
        S = L if train and L > 1 else _log(rng, 256, 8192)
        if B * L * S > 1 << 24:
            S = max(64, (1 << 24) // (B * L))
        return {"kind": kind, "B": B, "L": L, "S": S, "H": rng.choice([1, 2, 4, 4, 8]), "d": rng.choice([32, 64, 128, 128, 192]),
                "x": x, "train": train}
    return {"kind": kind, "T": _log(rng, 64, 32768), "K": _dim(rng, 128, 2048), "N": _dim(rng, 128, 4096),
            "E": rng.choice([4, 8, 16, 32]), "x": x, "w": w}


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------
class _Draws:
    def __init__(self, seed):
        self.g = torch.Generator(device="cuda").manual_seed(seed)

    def normal(self, *shape, std=1.0, dtype=F32):
        return (torch.randn(*shape, device="cuda", generator=self.g) * std).to(dtype)

    def activations(self, M, K, dtype):
        """N(0, 1) with 1% of the entries 20 times as large, as outlier channels make them."""
        t = torch.randn(M, K, device="cuda", generator=self.g)
        return torch.where(torch.rand(M, K, device="cuda", generator=self.g) < 0.01, t * 20, t).to(dtype)

    def routing(self, T, E, k):
        """Distinct experts per token with Zipf(1.1) popularity, and gates that sum to one."""
        p = torch.arange(1, E + 1, device="cuda", dtype=F32).pow(-1.1)
        idx = torch.multinomial(p.expand(T, E), k, replacement=False, generator=self.g)
        s = torch.sigmoid(torch.randn(T, k, device="cuda", generator=self.g))
        return idx, s / s.sum(-1, keepdim=True)


def _linear_inputs(c, seed):
    r = _Draws(seed)
    x = r.activations(c["M"], c["K"], _DT[c["x"]])
    w = r.normal(c["N"], c["K"], std=0.02, dtype=_DT[c["w"]])
    # FP8Linear's output is bf16, so its gradient is
    dy = r.normal(c["M"], c["N"], std=1e-3, dtype=BF16) if c["kind"] == "linear" else None
    return x, w, dy


def _experts_inputs(c, seed):
    r = _Draws(seed)
    x = r.normal(c["T"], c["D"], dtype=_DT[c["x"]])
    idx, scores = r.routing(c["T"], c["E"], c["k"])
    w12 = r.normal(c["E"], 2 * c["H"], c["D"], std=0.02)
    w3 = r.normal(c["E"], c["D"], c["H"], std=0.02)
    dout = r.normal(c["T"], c["D"], std=1e-2) if c["kind"] == "experts" else None
    return x, idx, scores, w12, w3, dout


def _indexer_inputs(c, seed):
    r = _Draws(seed)
    q = r.normal(c["B"], c["L"], c["H"], c["d"], dtype=_DT[c["x"]])
    k = r.normal(c["B"], c["S"], c["d"], dtype=_DT[c["x"]])
    w = r.normal(c["B"], c["L"], c["H"], std=0.5)
    g = r.normal(c["B"], c["L"], c["S"], std=1e-3) if c["train"] else None
    return q, k, w, g


def _grouped_inputs(c, seed):
    r = _Draws(seed)
    x = r.normal(c["T"], c["K"], dtype=_DT[c["x"]])
    w = r.normal(c["E"], c["N"], c["K"], std=0.02, dtype=_DT[c["w"]])
    idx, _ = r.routing(c["T"], c["E"], 1)
    ends = torch.bincount(idx.reshape(-1), minlength=c["E"]).cumsum(0)
    starts = torch.cat([ends.new_zeros(1), ends[:-1]])
    return x, w, starts, ends


def prepare(case, seed):
    kind = case["kind"]
    s = {"case": case}
    if kind in ("linear", "linear_infer"):
        x, w, s["dy"] = _linear_inputs(case, seed)
        lin = kernels.FP8Linear(128, 128, round_scale=case["round_scale"])
        lin.in_features, lin.out_features, lin.weight = case["K"], case["N"], torch.nn.Parameter(w)
        s["layer"], s["x"] = lin, x.requires_grad_(kind == "linear")
        if kind == "linear_infer":
            kernels.set_weight_cache(lin)
            with torch.no_grad():
                lin(torch.zeros_like(x))  # a serving program's warm-up fills the weight cache
    elif kind in ("experts", "experts_infer"):
        x, s["idx"], scores, w12, w3, s["dout"] = _experts_inputs(case, seed)
        ex = layers.GroupedExperts(1, 8, 8)
        ex.n_experts, ex.d_model, ex.hidden_dim = case["E"], case["D"], case["H"]
        ex.w12, ex.w3 = torch.nn.Parameter(w12), torch.nn.Parameter(w3)
        s["layer"] = ex
        s["x"], s["scores"] = x.requires_grad_(kind == "experts"), scores.requires_grad_(kind == "experts")
        if kind == "experts_infer":
            kernels.set_weight_cache(ex)
            ex.quantized_weights()
    elif kind == "indexer":
        s["q"], s["k"], w, s["g"] = _indexer_inputs(case, seed)
        s["w"], s["scale"] = w.requires_grad_(case["train"]), case["d"] ** -0.5
    elif kind == "grouped_f16":
        s["x"], s["w"], s["starts"], s["ends"] = _grouped_inputs(case, seed)
    else:
        s["x"], s["w"], _ = _linear_inputs(case, seed)
    return s


# ---------------------------------------------------------------------------
# One pass
# ---------------------------------------------------------------------------
def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "linear":
        lin = state["layer"]
        y = lin(state["x"])
        dx, dw = torch.autograd.grad(y, [state["x"], lin.weight], state["dy"])
        return {"y": y.detach(), "dx": dx, "dw": dw}
    if kind == "linear_infer":
        with torch.no_grad():
            return state["layer"](state["x"])
    if kind == "experts":
        ex = state["layer"]
        out, counts = moe.routed_experts(ex, state["x"], state["idx"], state["scores"])
        g = torch.autograd.grad(out, [state["x"], ex.w12, ex.w3, state["scores"]], state["dout"])
        return {"out": out.detach(), "counts": counts, "dx": g[0], "dw12": g[1], "dw3": g[2], "dscores": g[3]}
    if kind == "experts_infer":
        with torch.no_grad():
            out, counts = moe.routed_experts(state["layer"], state["x"], state["idx"], state["scores"])
        return {"out": out, "counts": counts}
    if kind == "indexer":
        scores = kernels.indexer_scores_fp8(state["q"], state["k"], state["w"], state["scale"])
        if not case["train"]:
            return {"scores": scores}
        (dw,) = torch.autograd.grad(scores, [state["w"]], state["g"])
        return {"scores": scores.detach(), "dw": dw}
    if kind == "grouped_f16":
        return kernels.moe_grouped_gemm(state["x"], state["w"], state["starts"], state["ends"])
    xq, xs = kernels.quantize_fp8_rowwise(state["x"], round_scale=case["round_scale"])
    wq, ws = kernels.quantize_fp8_blockwise(state["w"])
    if kind == "quantize":
        return {"xq": xq, "xs": xs, "wq": wq, "ws": ws}
    return kernels.fp8_matmul_dsv3(xq, wq.t().contiguous(), xs, ws.t().contiguous())


# ---------------------------------------------------------------------------
# What a pass cannot do without
# ---------------------------------------------------------------------------
_ES = {"bf16": 2, "fp16": 2, "fp32": 4}


def work(case):
    c, kind = case, case["kind"]
    es = _ES[c["x"]]
    if kind in ("linear", "linear_infer", "matmul", "quantize"):
        M, K, N = c["M"], c["K"], c["N"]
        cb = math.ceil(K / 128)
        if kind == "linear":
            b = M * K * es + N * K * _ES[c["w"]] + 2 * M * N + 2 * M * N + M * K * es + N * K * _ES[c["w"]]
            return {"bytes": b, "flops": 6 * M * K * N}
        if kind == "linear_infer":
            return {"bytes": M * K * es + N * K + math.ceil(N / 128) * cb * 4 + 2 * M * N, "flops": 2 * M * K * N}
        if kind == "matmul":
            return {"bytes": M * K * es + N * K * _ES[c["w"]] + 2 * M * N, "flops": 2 * M * K * N}
        return {"bytes": M * K * (es + 1) + 4 * M * cb + N * K * (_ES[c["w"]] + 1) + 4 * math.ceil(N / 128) * cb,
                "flops": 0}
    if kind in ("experts", "experts_infer"):
        T, D, H, E, k = c["T"], c["D"], c["H"], c["E"], c["k"]
        A = T * k
        io = T * D * es + A * 12 + 4 * T * D + 8 * E
        if kind == "experts":
            return {"bytes": io + 2 * E * 3 * H * D * 4 + 4 * T * D + T * D * es + 4 * A, "flops": 3 * 2 * A * 3 * H * D}
        # the experts that the tokens reach, their codes read once
        p = [(e + 1) ** -1.1 for e in range(E)]
        used = sum(1 - (1 - min(1.0, k * v / sum(p))) ** T for v in p)
        return {"bytes": int(io + used * 3 * H * D), "flops": 2 * A * 3 * H * D}
    if kind == "indexer":
        B, L, S, H, d = c["B"], c["L"], c["S"], c["H"], c["d"]
        b, f = B * (L * H * d + S * d) * es + 4 * B * L * H + 4 * B * L * S, 2 * B * L * S * H * d
        return {"bytes": b + 4 * B * L * S + 4 * B * L * H, "flops": 2 * f} if c["train"] else {"bytes": b, "flops": f}
    T, K, N, E = c["T"], c["K"], c["N"], c["E"]
    return {"bytes": T * K * es + E * N * K * _ES[c["w"]] + 2 * T * N, "flops": 2 * T * K * N}


def tolerance(case):
    return {
        # bf16 outputs: round to nearest gives 1.7e-3 of the norm and at most 2^-8 of a value
        "linear": {"rel": 7e-3, "max": 2e-2},
        "linear_infer": {"rel": 7e-3, "max": 2e-2},
        "matmul": {"rel": 7e-3, "max": 2e-2},
        # two quantized products in a chain: a rounding of the hidden values in 16 bits moves a
        # few of them by one e4m3 step
        "experts": {"rel": 1e-2, "max": 0.5},
        "experts_infer": {"rel": 1e-2, "max": 0.5},
        # fp32 sums of exact products in the matrix unit's internal order
        "indexer": {"rel": 6e-5, "max": 1e-3},
        "grouped_f16": {"rel": 8e-4, "max": 4e-3},
        "quantize": "exact",
    }[case["kind"]]


# ---------------------------------------------------------------------------
# The same results in plain torch, products in 64 bits
# ---------------------------------------------------------------------------
_FLOOR = torch.tensor(1e-4, dtype=F32).item()


def _quant_tiles(t, round_scale):
    """e4m3 codes and scale of tiles t [..., n]: scale = max(amax, 1e-4) / 448 in fp32 (rounded
    up to a power of two where asked), code = RNE(t / scale)."""
    t = t.float()
    s = (t.abs().amax(-1, keepdim=True).clamp(min=_FLOOR).double() / 448).float()
    if round_scale:
        m, e = torch.frexp(s)
        s = torch.ldexp(torch.ones_like(s), torch.where(m == 0.5, e - 1, e))
    # a 64-bit quotient rounded to 32 bits is the correctly rounded 32-bit quotient
    q = (t.double() / s.double()).float().clamp(-448, 448).to(torch.float8_e4m3fn)
    return q, s


def _quant_rows(t, round_scale=False):
    M, K = t.shape
    nb = -(-K // 128)
    q, s = _quant_tiles(torch.nn.functional.pad(t, (0, nb * 128 - K)).view(M, nb, 128), round_scale)
    return q.view(M, nb * 128)[:, :K], s.view(M, nb)


def _quant_blocks(t):
    M, K = t.shape
    bm, bk = -(-M // 128), -(-K // 128)
    v = torch.nn.functional.pad(t, (0, bk * 128 - K, 0, bm * 128 - M)).view(bm, 128, bk, 128).transpose(1, 2)
    q, s = _quant_tiles(v.reshape(bm, bk, 128 * 128), False)
    return q.view(bm, bk, 128, 128).transpose(1, 2).reshape(bm * 128, bk * 128)[:M, :K], s.view(bm, bk)


def _spread(s, n, dim):
    return s.repeat_interleave(128, dim).narrow(dim, 0, n)


def _rows(t, round_scale=False, dtype=torch.float64):
    """t after 1 x 128 quantization, widened."""
    q, s = _quant_rows(t, round_scale)
    return q.to(dtype) * _spread(s, t.shape[1], 1).to(dtype)


def _blocks(t):
    """t after 128 x 128 quantization, widened."""
    q, s = _quant_blocks(t)
    return q.double() * _spread(_spread(s, t.shape[1], 1), t.shape[0], 0).double()


def _cols(t, round_scale=False):
    """t after quantization in 128-row column tiles, widened."""
    return _rows(t.t().contiguous(), round_scale).t()


def _exact_experts(c, seed):
    x, idx, scores, w12, w3, dout = _experts_inputs(c, seed)
    T, D, H, E, k = c["T"], c["D"], c["H"], c["E"], c["k"]
    train = dout is not None
    flat = idx.reshape(-1)
    out = torch.zeros(T, D, dtype=torch.float64, device="cuda")
    r = {"out": out, "counts": torch.bincount(flat, minlength=E)}
    if train:
        r["dx"] = torch.zeros_like(out)
        r["dw12"] = torch.zeros(E, 2 * H, D, dtype=torch.float64, device="cuda")
        r["dw3"] = torch.zeros(E, D, H, dtype=torch.float64, device="cuda")
        r["dscores"] = torch.zeros(T * k, dtype=torch.float64, device="cuda")
    for e in range(E):
        at = (flat == e).nonzero().reshape(-1)
        if at.numel() == 0:
            continue
        tok, gate = at // k, scores.reshape(-1)[at, None]
        w12d, w3d = _blocks(w12[e]), _blocks(w3[e])
        xe = _rows(x[tok])
        # a value that is stored in 16 bits before the next quantization is rounded to them
        h12 = (xe @ w12d.t()).to(BF16).double()
        h1, h2 = h12[:, :H], h12[:, H:]
        he = _rows((torch.nn.functional.silu(h1) * h2).float().to(x.dtype))
        ye = he @ w3d.t()
        out.index_add_(0, tok, ye * gate)
        if not train:
            continue
        g = dout[tok]
        r["dscores"][at] = (g * ye).sum(-1)
        dy = (g * gate).to(BF16)
        dh = _rows(dy) @ w3d
        r["dw3"][e] = _cols(dy).t() @ _blocks(he.float())
        sig = torch.sigmoid(h1)
        d12 = torch.cat([dh * h2 * (sig * (1 + h1 * (1 - sig))), dh * (h1 * sig)], -1).float()
        r["dx"].index_add_(0, tok, _rows(d12) @ w12d)
        r["dw12"][e] = _cols(d12).t() @ _blocks(xe.float())
    if train:
        r["dscores"] = r["dscores"].view(T, k)
    return r


def exact(case, seed):
    c, kind = case, case["kind"]
    if kind in ("linear", "linear_infer", "matmul", "quantize"):
        x, w, dy = _linear_inputs(c, seed)
        rs = c["round_scale"]
        if kind == "quantize":
            (xq, xs), (wq, ws) = _quant_rows(x, rs), _quant_blocks(w)
            return {"xq": xq, "xs": xs, "wq": wq, "ws": ws}
        xd, wd = _rows(x, rs), _blocks(w)
        y = xd @ wd.t()
        if kind != "linear":
            return y
        xb = _blocks(_rows(x, rs, F32))
        return {"y": y, "dx": _rows(dy, rs) @ wd, "dw": _cols(dy, rs).t() @ xb}
    if kind in ("experts", "experts_infer"):
        return _exact_experts(c, seed)
    if kind == "indexer":
        q, k, w, g = _indexer_inputs(c, seed)
        B, L, S, H, d = c["B"], c["L"], c["S"], c["H"], c["d"]
        (q8, qs), (k8, ks) = _quant_rows(q.reshape(-1, d)), _quant_rows(k.reshape(-1, d))
        qs, ks = qs[:, 0].view(B, L, H).double(), ks[:, 0].view(B, 1, S).double()
        logits = q8.double().reshape(B, L * H, d) @ k8.double().reshape(B, S, d).transpose(1, 2).contiguous()
        logits = logits.relu_().view(B, L, H, S)
        scale = d ** -0.5
        out = {"scores": torch.zeros(B, L, S, dtype=torch.float64, device="cuda")}
        for h in range(H):
            out["scores"] += logits[:, :, h] * (qs[:, :, h] * w[:, :, h].double() * scale).unsqueeze(-1)
        out["scores"] *= ks
        if g is not None:
            gk = g.double() * ks
            out["dw"] = torch.stack([(logits[:, :, h] * gk).sum(-1) for h in range(H)], -1) * scale * qs
        return out
    x, w, starts, ends = _grouped_inputs(c, seed)
    out = torch.zeros(c["T"], c["N"], dtype=torch.float64, device="cuda")
    for e, (a, b) in enumerate(zip(starts.tolist(), ends.tolist())):
        out[a:b] = x[a:b].to(F16).double() @ w[e].to(F16).double().t()
    return out
