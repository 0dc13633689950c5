"""Performance cases of the LaplacianFormer operators on one GPU.

Three kinds of call, each through its public entry point:
  l1      LaplaceSubtraction forward and backward on the drop-in module, the backward
          either fused (LaplaceSubtraction_backward) or as the reference's two calls
          (backward_query, backward_key);
  newton  NewtonInverse forward and backward on the drop-in module, on the landmark
          Gram matrices exp(-L1(k, k) / sqrt(d)) + 1e-3 I that the attention inverts;
  layer   laplacian_attention through autograd: a training step (output and the
          gradients of q, k, v), or the output alone without gradients.

fp64 is left out: the operators take it for gradient checks, not for a model's work.
"""
from __future__ import annotations

import math

import torch

import laplacianformer_amd as lf

DTYPES = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
BYTES = {"f32": 4, "f16": 2, "bf16": 2}


def _l1(name, B, H, N, M, d, dtype, fused):
    return {"name": name, "kind": "l1", "B": B, "H": H, "N": N, "M": M, "d": d, "dtype": dtype, "fused": fused}


def _newton(name, mats, n, iters, dtype="f32"):
    return {"name": name, "kind": "newton", "mats": mats, "n": n, "iters": iters, "dtype": dtype}


def _layer(name, B, H, gh, gw, pool, d, dtype, train):
    return {"name": name, "kind": "layer", "B": B, "H": H, "gh": gh, "gw": gw, "pool": pool, "d": d, "iters": 10,
            "dtype": dtype, "train": train}


def listed():
    return [
        # A whole small layer in the default type: launches and host calls are what it costs.
        _layer("layer_tiny_f32", 2, 2, 14, 14, 2, 32, "f32", True),
        # The reference's own benchmark figure, N = M = 64 points, with its two backward calls.
        _l1("l1_pairs_f32", 32, 1, 64, 64, 64, "f32", False),
        # Distances of 56 x 56 tokens to 49 landmarks (first stage of a vision model), mixed precision.
        _l1("l1_stage1_f16", 32, 1, 3136, 49, 64, "f16", True),
        # The same stage trained in fp32 by a program written for the reference's module.
        _l1("l1_stage1_f32", 32, 1, 3136, 49, 64, "f32", False),
        # 55 x 55 tokens, 100 landmarks, 48 channels: sizes that fill no tile.
        _l1("l1_ragged_bf16", 12, 2, 3025, 100, 48, "bf16", True),
        # Many tokens and landmarks: the largest distance.
        _l1("l1_stress_bf16", 16, 8, 4096, 256, 64, "bf16", True),
        # The 7 x 7 landmarks' matrices of one stage: fewer matrices than the chip has CUs.
        _newton("newton_49", 32, 49, 10),
        # A batch of 64 x 64 matrices that fills the chip.
        _newton("newton_64", 1024, 64, 12),
        # The largest landmark sets that the inverse takes.
        _newton("newton_256", 128, 256, 16),
        # One training step of the layer at 28 x 28 tokens in mixed precision.
        _layer("layer_stage2_f16", 64, 2, 28, 28, 4, 64, "f16", True),
        # The layer at 56 x 56 tokens pooled 4 x 4: 196 landmarks.
        _layer("layer_stage1_bf16", 16, 1, 56, 56, 4, 64, "bf16", True),
        # A late stage, 14 x 14 tokens and four heads of 32 channels, in bf16.
        _layer("layer_stage3_bf16", 64, 4, 14, 14, 2, 32, "bf16", True),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["l1", "newton", "layer"])
    if kind == "l1":
        d = rng.choice([16, 24, 32, 40, 48, 64, 64, 96, 128, 50])
        M = rng.choice([49, 64, 128, _log_int(rng, 16, 256), _log_int(rng, 16, 256)])
        N = _log_int(rng, 16, 4096)
        H = rng.choice([1, 2, 3, 4, 8])
        # At most a quarter of the largest distance's work (odd channel counts run slower than whole vectors).
        most = max(1, int((2.0e9 if d % 8 == 0 else 4.0e8) // (H * N * M * d)))
        B = _log_int(rng, 1, min(64, most))
        c = _l1("", B, H, N, M, d, rng.choice(["f16", "bf16", "f32"]), rng.random() < 0.6)
    elif kind == "newton":
        n = rng.choice([49, 64, 100, 196, _log_int(rng, 12, 256), _log_int(rng, 12, 256)])
        iters = rng.randint(6, 16)
        most = max(1, int(1.2e11 // (4 * n ** 3 * iters)))
        c = _newton("", _log_int(rng, 4, min(1536, most)), n, iters)
    else:
        pool = rng.choice([2, 4, 4])
        mh, mw = rng.choice([(7, 7), (7, 7), (8, 8), (6, 9), (rng.randint(4, 14), rng.randint(4, 14))])
        d = rng.choice([24, 32, 48, 64, 64])
        H = rng.choice([1, 2, 4, 5])
        rows = H * mh * mw * pool * pool
        most = max(1, int(5.0e4 // rows)) if mh * mw > 64 else max(1, int(1.2e5 // rows))
        B = _log_int(rng, 1, min(64, most))
        c = _layer("", B, H, mh * pool, mw * pool, pool, d, rng.choice(["f16", "bf16", "f32"]), rng.random() < 0.75)
    del c["name"]
    return c


def _randn(gen, shape, dtype):
    return torch.randn(shape, generator=gen, device="cuda").to(dtype)


def _l1_pairs(x):
    """L1 distances of each set of points to itself, x [m, n, d] -> [m, n, n]."""
    out = torch.empty(x.shape[0], x.shape[1], x.shape[1], device=x.device, dtype=x.dtype)
    step = max(1, (1 << 27) // (x.shape[1] ** 2 * x.shape[2]))
    for i in range(0, x.shape[0], step):
        y = x[i:i + step]
        out[i:i + step] = (y[:, :, None] - y[:, None]).abs_().sum(-1)
    return out


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    t = DTYPES[case["dtype"]]
    if case["kind"] == "l1":
        B, H, N, M, d = (case[x] for x in ("B", "H", "N", "M", "d"))
        q, k, g = _randn(gen, (B, H, N, d), t), _randn(gen, (B, H, d, M), t), _randn(gen, (B, H, N, M), t)
        return {"case": case, "q": q, "k": k, "g": g, "out": torch.empty_like(g), "dq": torch.empty_like(q),
                "dk": torch.empty_like(k)}
    if case["kind"] == "newton":
        m, n = case["mats"], case["n"]
        dist = _l1_pairs(_randn(gen, (m, n, 64), torch.float32))
        a = (torch.exp(-dist / 8.0) + 1e-3 * torch.eye(n, device="cuda")).to(t).reshape(m, 1, n, n)
        return {"case": case, "a": a, "g": _randn(gen, (m, 1, n, n), t), "inv": torch.empty_like(a),
                "da": torch.empty_like(a)}
    shape = (case["B"], case["H"], case["gh"] * case["gw"], case["d"])
    q, k, v, g = (_randn(gen, shape, t) for _ in range(4))
    if case["train"]:
        for x in (q, k, v):
            x.requires_grad_()
    return {"case": case, "q": q, "k": k, "v": v, "g": g}


def run(s):
    case = s["case"]
    if case["kind"] == "l1":
        ops = lf.ext()
        q, k, g, out, dq, dk = (s[x] for x in ("q", "k", "g", "out", "dq", "dk"))
        ops.LaplaceSubtraction_forward(q, k, out)
        if case["fused"]:
            ops.LaplaceSubtraction_backward(g, q, k, dq, dk)
        else:
            ops.LaplaceSubtraction_backward_query(g, q, k, dq)
            ops.LaplaceSubtraction_backward_key(g, q, k, dk)
        return out, dq, dk
    if case["kind"] == "newton":
        ops = lf.ext()
        ops.NewtonInverse_forward(s["a"], s["inv"], case["iters"])
        ops.NewtonInverse_backward(s["g"], s["inv"], s["da"])
        return s["inv"], s["da"]
    q, k, v, grid = s["q"], s["k"], s["v"], (case["gh"], case["gw"])
    if not case["train"]:
        with torch.no_grad():
            return (lf.laplacian_attention(q, k, v, grid=grid, pool=case["pool"], iters=case["iters"]),)
    q.grad = k.grad = v.grad = None
    out = lf.laplacian_attention(q, k, v, grid=grid, pool=case["pool"], iters=case["iters"])
    out.backward(s["g"])
    return out.detach(), q.grad, k.grad, v.grad


def work(case):
    e = BYTES[case["dtype"]]
    if case["kind"] == "l1":
        BH, N, M, d = case["B"] * case["H"], case["N"], case["M"], case["d"]
        # q, k, g in; distances, dq, dk out. 3 flop per (row, landmark, channel) forward, 4 for each gradient.
        return {"bytes": 2 * e * BH * (N * d + M * d + N * M), "flops": 11 * BH * N * M * d}
    if case["kind"] == "newton":
        m, n = case["mats"], case["n"]
        return {"bytes": 4 * e * m * n * n, "flops": m * (case["iters"] + 1) * 4 * n ** 3}
    BH, N, d = case["B"] * case["H"], case["gh"] * case["gw"], case["d"]
    M = N // case["pool"] ** 2
    t = BH * (2 * N * M + M * M) * d            # triples of the three distances
    prod = 2 * BH * N * M * d                   # flops of one product of the N rows with the landmarks
    mm = 2 * BH * M * M * d
    inv = 4 * BH * M ** 3
    if not case["train"]:
        return {"bytes": 4 * e * BH * N * d, "flops": 3 * t + 2 * prod + mm + case["iters"] * inv}
    return {"bytes": 8 * e * BH * N * d, "flops": 11 * t + 6 * prod + 3 * mm + (case["iters"] + 1) * inv}


def tolerance(case):
    if case["kind"] == "l1":
        return {"rel": {"f32": 2e-6, "f16": 1e-3, "bf16": 8e-3}[case["dtype"]]}
    if case["kind"] == "newton":
        return {"rel": 2e-5}
    return {"rel": {"f32": 2e-5, "f16": 1.2e-3, "bf16": 1e-2}[case["dtype"]]}


def _distance_exact(q, k, g=None):
    """(distance, None, None), or with g the gradients of q and k too; q [m, N, d], k [m, d, M], fp64."""
    out = q.new_zeros(q.shape[0], q.shape[1], k.shape[2])
    dq, dk = (torch.empty_like(q), torch.empty_like(k)) if g is not None else (None, None)
    for c in range(q.shape[2]):
        diff = q[:, :, c, None] - k[:, c, None, :]
        out += diff.abs()
        if g is not None:
            diff.sign_().mul_(g)
            dq[:, :, c] = diff.sum(-1)
            dk[:, c] = -diff.sum(1)
    return out, dq, dk


def _inverse_exact(a, iters):
    p = a + 0.01 * torch.eye(a.shape[-1], device=a.device, dtype=a.dtype)
    v = p * (1.8 / p.sum(-1).amax(-1) ** 2)[:, None, None]
    for _ in range(iters):
        v = 2 * v - v @ (p @ v)
    return v


def _layer_exact(s):
    """The layer in 64 bits. The landmarks are rounded to the input type, as the layer defines them."""
    case = s["case"]
    B, H, gh, gw, p, d = (case[x] for x in ("B", "H", "gh", "gw", "pool", "d"))
    t, N = s["q"].dtype, gh * gw
    q, k, v, g = (s[x].detach().double().reshape(B * H, N, d) for x in ("q", "k", "v", "g"))
    km = k.reshape(B * H, gh // p, p, gw // p, p, d).mean(dim=(2, 4)).reshape(B * H, -1, d).to(t).double()
    key = km.transpose(1, 2).contiguous()
    sc = 1.0 / math.sqrt(d)
    kqm, kmm, kkm = (torch.exp(-sc * _distance_exact(x, key)[0]) for x in (q, km, k))
    inv = _inverse_exact(kmm, case["iters"])
    kv = kkm.transpose(1, 2) @ v
    w = inv @ kv
    out = kqm @ w
    shape = (B, H, N, d)
    if not case["train"]:
        return (out.reshape(shape),)
    dw = kqm.transpose(1, 2) @ g
    dkv = inv.transpose(1, 2) @ dw
    dmm = -(inv.transpose(1, 2) @ (dw @ kv.transpose(1, 2))) @ inv.transpose(1, 2)
    grads = [(q, g @ w.transpose(1, 2), kqm), (km, dmm, kmm), (k, v @ dkv.transpose(1, 2), kkm)]
    (dq, k1), (dkm, k2), (dk, k3) = (_distance_exact(x, key, -sc * gx * kx)[1:] for x, gx, kx in grads)
    dkm = (dkm + (k1 + k2 + k3).transpose(1, 2)) / (p * p)
    dkm = dkm.reshape(B * H, gh // p, 1, gw // p, 1, d).expand(-1, -1, p, -1, p, -1).reshape(B * H, N, d)
    return out.reshape(shape), dq.reshape(shape), (dk + dkm).reshape(shape), (kkm @ dkv).reshape(shape)


def exact(case, seed):
    s = prepare(case, seed)
    if case["kind"] == "layer":
        return _layer_exact(s)
    if case["kind"] == "newton":
        m, n = case["mats"], case["n"]
        v = _inverse_exact(s["a"].double().reshape(m, n, n), case["iters"])
        g, vt = s["g"].double().reshape(m, n, n), v.transpose(1, 2)
        return v.reshape(m, 1, n, n), -(vt @ g @ vt).reshape(m, 1, n, n)
    B, H = case["B"], case["H"]
    q, k, g = (s[x].double().flatten(0, 1) for x in ("q", "k", "g"))
    return tuple(x.unflatten(0, (B, H)) for x in _distance_exact(q, k, g))
