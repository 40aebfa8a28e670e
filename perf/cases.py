"""What the performance of this framework is measured on.

Every case is one call sequence of a program that fine-tunes or runs a
transformer through the framework's public entry points: LoRA linears in
inference (decode and prefill) and in training (forward and backward, float32
and bfloat16, single and grouped), the attention core, the norms, the softmax
of materialised scores and the loss. Sizes are those of the layers that
bench.py and the tests run, or odd and ragged ones of the same ranges (batches
padded to their longest sequence, prompts of any length).
"""
import math

import torch

import __graft_entry__

mc = __graft_entry__.load_package()

# Projection sizes [in, out] of the layers that bench.py and the tests run.
SMALL = [(768, 768), (896, 896), (896, 128)]
MEDIUM = [(1536, 1536), (1536, 256), (1536, 8960), (8960, 1536)]
LARGE = [(3584, 3584), (3584, 512), (3584, 18944), (18944, 3584)]
DTYPES = {"f32": torch.float32, "bf16": torch.bfloat16}
BYTES = {"f32": 4, "bf16": 2}


def listed():
    return [
        # One new token of one sequence through a square projection: the
        # smallest call, where launches and latency count.
        {"name": "lora_decode", "kind": "lora_infer", "T": 1, "K": 1536, "N": 1536, "r": 16, "bias": True},
        # A prompt of an arbitrary length through an MLP projection.
        {"name": "lora_prefill", "kind": "lora_infer", "T": 777, "K": 1536, "N": 8960, "r": 16, "bias": False},
        # A float32 LoRA linear of 4 x 128 tokens, one training step's forward
        # and backward.
        {"name": "lora_train_f32", "kind": "lora_train", "dtype": "f32", "T": 512, "K": 768, "N": 768, "r": 8,
         "p": 0.0, "bias": False},
        # Float32 fine-tuning of an MLP projection, four ragged sequences.
        {"name": "lora_train_f32_mlp", "kind": "lora_train", "dtype": "f32", "T": 4 * 509, "K": 1536, "N": 8960,
         "r": 16, "p": 0.0, "bias": False},
        # A bfloat16 attention projection called on its own, 16 x 512 tokens.
        {"name": "lora_train_bf16", "kind": "lora_train", "dtype": "bf16", "T": 16 * 512, "K": 896, "N": 896, "r": 8,
         "p": 0.0, "bias": True},
        # Gate and up projections of a 3584-wide layer as a group, rank 64 with
        # dropout, W^T laid out at load: the largest case.
        {"name": "lora_group_mlp", "kind": "lora_group", "T": 4 * 4096, "K": 3584, "Ns": "18944,18944", "r": 64,
         "p": 0.1},
        # The attention core of a training step.
        {"name": "attn_train_bf16", "kind": "attn", "dtype": "bf16", "B": 8, "H": 12, "Hkv": 2, "S": 2048, "D": 128,
         "causal": True, "train": True},
        # The attention core over one prompt of an arbitrary length.
        {"name": "attn_prefill_bf16", "kind": "attn", "dtype": "bf16", "B": 1, "H": 14, "Hkv": 2, "S": 777, "D": 64,
         "causal": True, "train": False},
        # Float32 attention of a training step, four ragged sequences.
        {"name": "attn_train_f32", "kind": "attn", "dtype": "f32", "B": 4, "H": 12, "Hkv": 2, "S": 509, "D": 64,
         "causal": True, "train": True},
        # The norm in front of a block, forward and backward.
        {"name": "norm_train_f32", "kind": "norm", "op": "rms", "dtype": "f32", "rows": 8192, "dim": 896},
        # Causal softmax over materialised scores of ragged sequences.
        {"name": "softmax_train_f32", "kind": "softmax", "dtype": "f32", "B": 4, "H": 14, "S": 777, "causal": True},
        # The loss over a vocabulary, prompt tokens ignored.
        {"name": "loss_train_bf16", "kind": "xent", "dtype": "bf16", "rows": 4 * 509, "V": 151936, "smoothing": 0.0},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["decode", "prefill", "lora_f32", "lora_bf16", "lora_group", "attn_bf16", "attn_prefill",
                       "attn_f32", "norm", "softmax", "xent"])
    if kind == "decode":  # a few sequences, one token each
        K, N = rng.choice(SMALL + MEDIUM + LARGE)
        return {"kind": "lora_infer", "T": _log_int(rng, 1, 64), "K": K, "N": N, "r": rng.choice([8, 16, 64]),
                "bias": rng.random() < 0.5}
    if kind == "prefill":
        K, N = rng.choice(SMALL + MEDIUM + LARGE)
        return {"kind": "lora_infer", "T": _log_int(rng, 65, 4096), "K": K, "N": N, "r": rng.choice([8, 16, 64]),
                "bias": rng.random() < 0.5}
    if kind == "lora_f32":
        K, N = rng.choice(SMALL + MEDIUM)
        return {"kind": "lora_train", "dtype": "f32", "T": _log_int(rng, 32, 4096), "K": K, "N": N,
                "r": rng.choice([4, 8, 16, 64]), "p": rng.choice([0.0, 0.1]), "bias": rng.random() < 0.5}
    if kind == "lora_bf16":
        K, N = rng.choice(SMALL + MEDIUM)
        return {"kind": "lora_train", "dtype": "bf16", "T": _log_int(rng, 128, 16384), "K": K, "N": N,
                "r": rng.choice([4, 8, 16, 64]), "p": rng.choice([0.0, 0.1]), "bias": rng.random() < 0.5}
    if kind == "lora_group":
        K, Ns = rng.choice([(896, "896,128,128"), (1536, "1536,256,256"), (1536, "8960,8960"), (3584, "3584,512,512"),
                            (3584, "18944,18944")])
        return {"kind": "lora_group", "T": _log_int(rng, 512, 16384), "K": K, "Ns": Ns, "r": rng.choice([8, 16, 64]),
                "p": rng.choice([0.0, 0.1])}
    if kind in ("attn_bf16", "attn_prefill"):
        H, Hkv, D = rng.choice([(14, 2, 64), (12, 2, 128), (28, 4, 128), (12, 12, 64)])
        train = kind == "attn_bf16"
        return {"kind": "attn", "dtype": "bf16", "B": rng.choice([1, 2, 3, 4, 8]) if train else 1, "H": H,
                "Hkv": Hkv, "S": _log_int(rng, 32, 2048), "D": D, "causal": rng.random() < 0.75, "train": train}
    if kind == "attn_f32":
        H, Hkv, D = rng.choice([(12, 12, 32), (14, 2, 64), (12, 2, 64), (12, 12, 64), (12, 2, 128)])
        return {"kind": "attn", "dtype": "f32", "B": rng.choice([1, 2, 3, 4]), "H": H, "Hkv": Hkv,
                "S": _log_int(rng, 16, 512), "D": D, "causal": rng.random() < 0.5, "train": rng.random() < 0.7}
    if kind == "norm":
        dim = _log_int(rng, 256, 4096)
        if rng.random() < 0.7:
            dim = (dim + 63) // 64 * 64
        return {"kind": "norm", "op": rng.choice(["rms", "layer"]), "dtype": rng.choice(["f32", "bf16"]),
                "rows": _log_int(rng, 64, 16384), "dim": dim}
    if kind == "softmax":
        return {"kind": "softmax", "dtype": rng.choice(["f32", "bf16"]), "B": rng.choice([1, 2, 4, 8]),
                "H": rng.choice([12, 14]), "S": _log_int(rng, 32, 1024), "causal": rng.random() < 0.75}
    return {"kind": "xent", "dtype": rng.choice(["f32", "bf16"]), "rows": _log_int(rng, 64, 4096),
            "V": rng.choice([_log_int(rng, 1000, 151936), 151936]), "smoothing": rng.choice([0.0, 0.1])}


# ------------------------------------------------------------------ inputs
def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _normal(g, shape, std=1.0, mean=0.0, dtype=torch.float32):
    t = torch.empty(shape, dtype=torch.float32, device="cuda")
    return t.normal_(mean, std, generator=g).to(dtype)


def _factors(g, K, N, r):
    """A kaiming-uniform [K, r] and a trained B ~ N(0, 0.02) [r, N], float32."""
    A = torch.empty(K, r, device="cuda").uniform_(-K ** -0.5, K ** -0.5, generator=g)
    return A, _normal(g, (r, N), 0.02)


def _mask(g, T, r, p):
    if p == 0.0:
        return None
    return (torch.empty(T, r, device="cuda").uniform_(0.0, 1.0, generator=g) >= p).to(torch.uint8)


def _inputs(case, seed):
    g = _gen(seed)
    kind = case["kind"]
    if kind in ("lora_infer", "lora_train"):
        T, K, N, r = case["T"], case["K"], case["N"], case["r"]
        dt = DTYPES[case.get("dtype", "bf16")]
        s = {"x": _normal(g, (T, K), dtype=dt), "W": _normal(g, (N, K), 0.02, dtype=dt)}
        s["A"], s["B"] = _factors(g, K, N, r)
        s["bias"] = _normal(g, (N,), 0.02, dtype=dt) if case["bias"] else None
        if kind == "lora_train":
            s["dY"] = _normal(g, (T, N), 1e-2, dtype=dt)
            s["mask"] = _mask(g, T, r, case["p"])
        return s
    if kind == "lora_group":
        T, K, r = case["T"], case["K"], case["r"]
        dt = torch.bfloat16
        s = {"x": _normal(g, (T, K), dtype=dt), "projs": [], "dYs": []}
        for N in _outs(case):
            A, B = _factors(g, K, N, r)
            s["projs"].append({"W": _normal(g, (N, K), 0.02, dtype=dt), "bias": None, "A": A, "B": B,
                               "mask": _mask(g, T, r, case["p"])})
            s["dYs"].append(_normal(g, (T, N), 1e-2, dtype=dt))
        return s
    if kind == "attn":
        B, H, Hkv, S, D = (case[k] for k in ("B", "H", "Hkv", "S", "D"))
        dt = DTYPES[case["dtype"]]
        s = {"q": _normal(g, (B, H, S, D), dtype=dt), "k": _normal(g, (B, Hkv, S, D), dtype=dt),
             "v": _normal(g, (B, Hkv, S, D), dtype=dt)}
        if case["train"]:
            s["dout"] = _normal(g, (B, S, H * D), 1e-2, dtype=dt)
        return s
    if kind == "norm":
        rows, dim, dt = case["rows"], case["dim"], DTYPES[case["dtype"]]
        return {"x": _normal(g, (rows, dim), dtype=dt), "w": _normal(g, (dim,), 0.1, 1.0, dtype=dt),
                "b": _normal(g, (dim,), 0.1, dtype=dt), "dy": _normal(g, (rows, dim), 1e-2, dtype=dt)}
    if kind == "softmax":
        shape, dt = (case["B"], case["H"], case["S"], case["S"]), DTYPES[case["dtype"]]
        return {"s": _normal(g, shape, 3.0, dtype=dt), "dp": _normal(g, shape, 1e-2, dtype=dt)}
    rows, V = case["rows"], case["V"]
    targets = torch.randint(0, V, (rows,), generator=g, device="cuda", dtype=torch.int32)
    targets[: rows // 4] = IGNORE  # the prompt's tokens carry no loss
    return {"logits": _normal(g, (rows, V), 2.0, dtype=DTYPES[case["dtype"]]), "targets": targets}


IGNORE = 0  # the padding token's id


def _outs(case):
    return [int(n) for n in case["Ns"].split(",")]


def prepare(case, seed):
    s = _inputs(case, seed)
    s["case"] = case
    for proj in s.get("projs", []):  # the frozen W's transpose, built once at load
        proj["Wt"] = mc.transpose_weight(proj["W"])
    return s


SCALE = 2.0  # alpha / rank
EPS = 1e-6


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "lora_infer":
        return mc.lora_forward(s["x"], s["A"], s["B"], SCALE, W=s["W"], bias=s["bias"], save_hidden=False)[0]
    if kind == "lora_train":
        p = case["p"]
        y, h = mc.lora_forward(s["x"], s["A"], s["B"], SCALE, W=s["W"], bias=s["bias"], mask=s["mask"], dropout_p=p)
        return (y,) + mc.lora_backward(s["x"], s["A"], s["B"], s["dY"], SCALE, W=s["W"], mask=s["mask"], dropout_p=p,
                                       h_save=h)
    if kind == "lora_group":
        p = case["p"]
        ys, hs = mc.lora_group_forward(s["x"], s["projs"], SCALE, dropout_p=p)
        dX, dAs, dBs = mc.lora_group_backward(s["x"], s["projs"], s["dYs"], SCALE, dropout_p=p, h_saves=hs)
        return [*ys, dX, *dAs, *dBs]
    if kind == "attn":
        o, lse = mc.attention_forward(s["q"], s["k"], s["v"], causal=case["causal"], save_lse=case["train"])
        if not case["train"]:
            return o
        return (o, lse) + mc.attention_backward(s["q"], s["k"], s["v"], o, lse, s["dout"], causal=case["causal"])
    if kind == "norm":
        if case["op"] == "rms":
            y, rstd = mc.rms_norm_forward(s["x"], EPS, s["w"])
            return (y,) + mc.rms_norm_backward(s["x"], s["dy"], EPS, s["w"], rstd)
        y, mean, rstd = mc.layer_norm_forward(s["x"], EPS, s["w"], s["b"])
        return (y,) + mc.layer_norm_backward(s["x"], s["dy"], EPS, s["w"], mean, rstd)
    if kind == "softmax":
        causal = case["S"] if case["causal"] else 0
        p = mc.softmax_forward(s["s"], causal)
        return p, mc.softmax_backward(p, s["dp"], causal)
    loss, stats = mc.cross_entropy_forward(s["logits"], s["targets"], IGNORE, case["smoothing"])
    return loss, mc.cross_entropy_backward(s["logits"], s["targets"], stats, None, IGNORE, case["smoothing"])


# -------------------------------------------------------------------- work
def _lora_work(T, K, N, r, es, train, masked):
    flops = 2.0 * T * K * N + 2.0 * T * r * (K + N)
    data = es * (T * K + N * K + T * N) + 4 * r * (K + N)
    if train:
        flops = 2 * flops + 2.0 * T * r * (K + N)  # dX with its rank-r terms, then dA and dB
        data += es * (T * N + T * K) + 4 * r * (K + N) + (T * r if masked else 0)
    return data, flops


def work(case):
    kind = case["kind"]
    if kind in ("lora_infer", "lora_train"):
        data, flops = _lora_work(case["T"], case["K"], case["N"], case["r"], BYTES[case.get("dtype", "bf16")],
                                 kind == "lora_train", case.get("p", 0.0) > 0)
        return {"bytes": data, "flops": flops}
    if kind == "lora_group":
        parts = [_lora_work(case["T"], case["K"], N, case["r"], 2, True, case["p"] > 0) for N in _outs(case)]
        shared = 2 * 2 * case["T"] * case["K"] * (len(parts) - 1)  # one x and one dX for the group
        return {"bytes": sum(d for d, _ in parts) - shared, "flops": sum(f for _, f in parts)}
    if kind == "attn":
        B, H, Hkv, S, D = (case[k] for k in ("B", "H", "Hkv", "S", "D"))
        pairs = B * H * (S * (S + 1) / 2 if case["causal"] else S * S)
        qo, kv = B * H * S * D, B * Hkv * S * D
        if not case["train"]:
            return {"bytes": BYTES[case["dtype"]] * (2 * qo + 2 * kv), "flops": 4.0 * pairs * D}
        return {"bytes": BYTES[case["dtype"]] * (4 * qo + 4 * kv) + 4 * B * H * S, "flops": 14.0 * pairs * D}
    if kind == "norm":
        n = case["rows"] * case["dim"]
        return {"bytes": 4 * n * BYTES[case["dtype"]], "flops": 16.0 * n}
    if kind == "softmax":
        S = case["S"]
        whole = case["B"] * case["H"] * S * S
        read = case["B"] * case["H"] * S * (S + 1) // 2 if case["causal"] else whole
        return {"bytes": BYTES[case["dtype"]] * 2 * (read + whole), "flops": 8.0 * read}
    n = case["rows"] * case["V"]
    return {"bytes": 2 * n * BYTES[case["dtype"]], "flops": 6.0 * n}


def tolerance(case):
    # About four times the largest relative distance from `exact` seen on any
    # output over the listed and two dozen drawn cases. bfloat16: 2.5e-3, the
    # rounding of the outputs and of the operands between two products.
    # float32: 1e-6 for the products (the order of long sums), 3e-7 for the
    # row operations.
    if case.get("dtype", "bf16") == "bf16":
        return {"rel": 1e-2}
    return {"rel": 5e-6 if case["kind"] in ("lora_train", "attn") else 1.5e-6}


# ------------------------------------------------------------------- exact
def _lora_exact(x, proj, dY, mask, p):
    A, B, W = (proj[k].double() for k in ("A", "B", "W"))
    keep = 1.0 if mask is None else mask.double() / (1.0 - p)
    h = (x @ A) * keep
    y = x @ W.t() + SCALE * (h @ B)
    if proj.get("bias") is not None:
        y += proj["bias"].double()
    if dY is None:
        return y
    g = SCALE * (dY @ B.t()) * keep
    return y, dY @ W + g @ A.t(), x.t() @ g, SCALE * (h.t() @ dY)


def exact(case, seed):
    s = _inputs(case, seed)
    kind = case["kind"]
    if kind == "lora_infer":
        return _lora_exact(s["x"].double(), s, None, None, 0.0)
    if kind == "lora_train":
        return _lora_exact(s["x"].double(), s, s["dY"].double(), s["mask"], case["p"])
    if kind == "lora_group":
        outs = [_lora_exact(s["x"].double(), proj, dY.double(), proj["mask"], case["p"])
                for proj, dY in zip(s["projs"], s["dYs"])]
        return [*(o[0] for o in outs), sum(o[1] for o in outs), *(o[2] for o in outs), *(o[3] for o in outs)]
    if kind == "attn":
        return _attn_exact(case, s)
    if kind == "norm":
        x, w, dy = s["x"].double(), s["w"].double(), s["dy"].double()
        if case["op"] == "layer":
            x = x - x.mean(-1, keepdim=True)
        rstd = (x.square().mean(-1, keepdim=True) + EPS).rsqrt()
        xh = x * rstd
        g = dy * w
        dx = g - xh * (g * xh).mean(-1, keepdim=True)
        if case["op"] == "layer":
            dx = dx - g.mean(-1, keepdim=True)
            return xh * w + s["b"].double(), dx * rstd, (dy * xh).sum(0), dy.sum(0)
        return xh * w, dx * rstd, (dy * xh).sum(0)
    if kind == "softmax":
        x = s["s"].double()
        if case["causal"]:
            S = case["S"]
            x = x.masked_fill(torch.ones(S, S, dtype=torch.bool, device="cuda").triu(1), float("-inf"))
        p = torch.softmax(x, -1)
        dp = s["dp"].double()
        return p, p * (dp - (p * dp).sum(-1, keepdim=True))
    x, t = s["logits"].double(), s["targets"].long()
    V, eps = case["V"], case["smoothing"]
    counted = t != IGNORE
    n = counted.sum()
    lp = torch.log_softmax(x, -1)
    nll = -lp.gather(1, t[:, None])[:, 0][counted].sum() / n
    # the smoothing term averages over every row, as the reference's does
    loss = (1.0 - eps) * nll + eps * -lp.mean()
    probs = lp.exp_()
    onehot = torch.zeros_like(probs).scatter_(1, t[:, None], 1.0)
    dlogits = (1.0 - eps) * (probs - onehot) * counted[:, None] / n
    dlogits += eps * (probs - 1.0 / V) / case["rows"]
    return loss.reshape(1), dlogits


def _attn_exact(case, s):
    B, H, Hkv, S, D = (case[k] for k in ("B", "H", "Hkv", "S", "D"))
    rep, scale = H // Hkv, D ** -0.5
    above = torch.ones(S, S, dtype=torch.bool, device="cuda").triu(1) if case["causal"] else None
    o = torch.empty(B, S, H, D, dtype=torch.float64, device="cuda")
    lse = torch.empty(B, H, S, dtype=torch.float64, device="cuda")
    dq = torch.zeros(B, H, S, D, dtype=torch.float64, device="cuda")
    dk = torch.zeros(B, Hkv, S, D, dtype=torch.float64, device="cuda")
    dv = torch.zeros_like(dk)
    dout = s["dout"].double().reshape(B, S, H, D) if case["train"] else None
    for b in range(B):
        for h in range(H):
            q, k, v = s["q"][b, h].double(), s["k"][b, h // rep].double(), s["v"][b, h // rep].double()
            sc = (q @ k.t()) * scale
            if above is not None:
                sc = sc.masked_fill(above, float("-inf"))
            lse[b, h] = torch.logsumexp(sc, -1)
            p = torch.softmax(sc, -1)
            o[b, :, h] = p @ v
            if case["train"]:
                do = dout[b, :, h]
                dv[b, h // rep] += p.t() @ do
                ds = p * (do @ v.t() - (do * o[b, :, h]).sum(-1, keepdim=True))
                dq[b, h] = (ds @ k) * scale
                dk[b, h // rep] += (ds.t() @ q) * scale
    o = o.reshape(B, S, H * D)
    return (o, lse, dq, dk, dv) if case["train"] else o
