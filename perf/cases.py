"""Performance cases of the quantization path: what a build, a measure step or a table fit calls, through the
package's own entry points.

    listed()            the cases, dicts of plain values
    draw(rng)           one more case of the same ranges
    prepare(case, seed) what a program holds before the call (inputs from the seed; plans, tables, factors it keeps)
    run(state)          one pass, its outputs whole
    work(case)          bytes and operations one pass cannot do without
    tolerance(case)     how far another correct implementation at the same precision may be off
    exact(case, seed)   the same outputs in 64 bits, by plain torch
"""

from __future__ import annotations

import math

import torch

from lookatmyquant_amd import codes, compiler, engine, ldlq_gpu, quantize, tables
from lookatmyquant_amd.frame import Environment

DEV = "cuda"
HEAD = 128  # head dim of the forwards' attention


def listed() -> list[dict]:
    return [
        # The calibration forwards' attention of a layer (32 query, 8 key/value heads), a quarter of the benchmark's
        # 32 sequences: the largest kernel of a layer's forwards.
        {"name": "attention_8x2048", "kind": "attention", "B": 8, "T": 2048, "heads": 32, "kv": 8},
        # One short prompt of an odd length, as an evaluation window: few workgroups, the launch counts.
        {"name": "attention_1x333", "kind": "attention", "B": 1, "T": 333, "heads": 32, "kv": 8},
        # The passes around a layer's matrix products on four sequences: the padded input norm, q's per-head norm
        # with the rotary embedding, and the SwiGLU gate.
        {"name": "pointwise_4x2048", "kind": "pointwise", "B": 4, "T": 2048, "hidden": 2560, "heads": 32,
         "inter": 9728},
        # A stage's statistics: the digit-weighted Hessian and the cross-Gram of both streams.
        {"name": "statistics_2560", "kind": "statistics", "N": 16384, "n": 2560, "weighted": True, "cross": True},
        # The environment of a linear layer of o_proj's width: the damped factor, its success checked.
        {"name": "factor_4096", "kind": "factor", "n": 4096},
        # The rotation of a stage's statistics into the incoherent basis.
        {"name": "rotation_4096", "kind": "rotation", "n": 4096},
        # The QEP targets of a gate/up/q/k/v stage: its own factor and three fp64 products.
        {"name": "qep_2560", "kind": "qep", "n": 2560, "m": 1024},
        # A stage's row groups at 1 to 4 bits on the fitted 12-bit trellis (the production build), q, k and v.
        {"name": "sweep_L12_6144x2560", "kind": "sweep", "L": 12, "n": 2560, "m": 6144, "bits": "23321234"},
        # The same at 16 state bits, one 960 x 960 matrix at the plan's mixed widths.
        {"name": "sweep_L16_960x960", "kind": "sweep", "L": 16, "n": 960, "m": 960, "bits": "232314"},
        # One 960 x 960 projection at 3 bits on Lloyd-Max levels.
        {"name": "lloyd_960x960", "kind": "lloyd", "n": 960, "m": 960, "levels": 8},
        # One batch of a trellis-table fit: 256 sequences of 256 samples, the first state free.
        {"name": "viterbi_256x256", "kind": "viterbi", "L": 12, "k": 2, "B": 256, "T": 256},
        # The measure step's KL over one window's logits at the benchmark's vocabulary.
        {"name": "kl_2048", "kind": "kl", "T": 2048, "V": 151936, "dtype": "bf16"},
    ]


def _log(rng, lo: int, hi: int) -> int:
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


WIDTHS = (256, 320, 512, 640, 960, 1280, 1536, 2048, 2560)  # orders the rotation has a Hadamard matrix for


def draw(rng) -> dict:
    kind = rng.choice(["attention", "pointwise", "statistics", "factor", "rotation", "qep", "sweep", "sweep", "lloyd",
                       "viterbi", "kl"])
    c: dict = {"kind": kind}
    if kind == "attention":
        kv = rng.choice([1, 2, 8])
        c |= {"T": _log(rng, 1, 2048), "heads": kv * rng.choice([1, 3, 4]), "kv": kv}
        c["B"] = _log(rng, 1, max(1, 16384 // max(64, c["T"])))
    elif kind == "pointwise":
        c |= {"B": rng.randint(1, 4), "T": _log(rng, 1, 2048), "hidden": rng.choice([960, 1024, 2560, 4096]),
              "heads": rng.choice([8, 15, 32]), "inter": rng.choice([2560, 4096, 9728])}
    elif kind == "statistics":
        c |= {"n": rng.choice([256, 960, 1000, 2560, 4096]), "weighted": rng.random() < 0.7,
              "cross": rng.random() < 0.6}
        c["N"] = _log(rng, 257, 16384 if c["n"] <= 2560 else 8192)
    elif kind == "factor":
        c["n"] = _log(rng, 64, 4096)
    elif kind == "rotation":
        c["n"] = rng.choice(WIDTHS + (4096,))
    elif kind == "qep":
        c["n"] = _log(rng, 128, 2560)
        c["m"] = _log(rng, 64, 2 * c["n"])
    elif kind == "sweep":
        c["L"] = rng.choice([12, 12, 16])
        c["n"] = rng.choice(WIDTHS[:-1] if c["L"] == 12 else WIDTHS[:5])
        most = (6144 * 2560 if c["L"] == 12 else 960 * 960) // c["n"]
        c["m"] = _log(rng, 33, min(most, 6144))
        c["bits"] = "".join(rng.choice("1223334") for _ in range(rng.randint(1, 8)))
    elif kind == "lloyd":
        c |= {"n": _log(rng, 128, 2560), "m": _log(rng, 17, 2048), "levels": rng.choice([2, 3, 4, 8, 16])}
    elif kind == "viterbi":
        c["L"] = rng.choice([8, 10, 12, 12, 16])
        c |= {"k": rng.randint(1, 4), "T": _log(rng, 8, 256)}
        c["B"] = _log(rng, 1, 1024 if c["L"] < 16 else 128)
    else:
        c |= {"T": _log(rng, 1, 2048), "V": rng.choice([151936, 151936, 49152, 32003]),
              "dtype": rng.choice(["bf16", "bf16", "f32"])}
        if c["dtype"] == "f32":
            c["T"] = max(1, c["T"] // 2)
    return c


# ----------------------------------------------------------------------------- inputs


def _gen(seed: int) -> torch.Generator:
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _randn(g, *shape, dtype=torch.float32):
    return torch.randn(*shape, generator=g, device=DEV, dtype=dtype)


def _activations(g, N: int, n: int, scale: torch.Tensor) -> torch.Tensor:
    """Channel-scaled Gaussian activations, bf16."""
    return (_randn(g, N, n) * scale).to(torch.bfloat16)


def _channels(g, n: int) -> torch.Tensor:
    """Heavy-tailed channel scales, as transformer activations have."""
    return torch.exp(0.5 * _randn(g, n))


def _statistics(g, n: int) -> torch.Tensor:
    """The float64 second moment of 2n + 256 channel-scaled tokens, through float32 as the Gram kernels leave it."""
    X = _randn(g, 2 * n + 256, n) * _channels(g, n)
    H = (X.T @ X / X.shape[0]).double()
    return ((H + H.T) / 2).contiguous()


def _digit_weights(g, N: int) -> torch.Tensor:
    """A tenth of the tokens weighted ten times the rest, mean 1."""
    w = torch.where(torch.rand(N, generator=g, device=DEV) < 0.1, 10.0, 1.0)
    return (w / w.mean()).float()


def _row_groups(seed: int, m: int, bits: str) -> list[dict]:
    """A random permutation of the rows cut evenly, one width per cut, as a row plan gives them."""
    perm = torch.randperm(m, generator=torch.Generator().manual_seed(int(seed))).tolist()
    cuts = [m * i // len(bits) for i in range(len(bits) + 1)]
    return [{"group": i, "rows": sorted(perm[cuts[i] : cuts[i + 1]]), "bits": int(b)}
            for i, b in enumerate(bits) if cuts[i + 1] > cuts[i]]


def _table(L: int, k: int) -> torch.Tensor:
    if L == 12:
        t = tables.load_table(12, k)
    else:
        t = tables.quantile_table(L, 0)
    return torch.tensor(t, dtype=torch.float64, device=DEV)


def _inputs(c: dict, seed: int) -> dict:
    """The case's inputs alone (no plan, table or factor)."""
    g, kind = _gen(seed), c["kind"]
    if kind == "attention":
        B, T, H, kv = c["B"], c["T"], c["heads"], c["kv"]
        # q and k after their per-head norm; the projections leave [B, T, heads, 128], passed transposed
        mk = lambda h: _randn(g, B, T, h, HEAD).to(torch.bfloat16).transpose(1, 2)
        return {"q": mk(H), "k": mk(kv), "v": mk(kv)}
    if kind == "pointwise":
        B, T = c["B"], c["T"]
        bf = lambda *s: _randn(g, *s).to(torch.bfloat16)
        ang = torch.outer(torch.arange(T, device=DEV, dtype=torch.float32),
                          1e6 ** (-torch.arange(0, HEAD, 2, device=DEV, dtype=torch.float32) / HEAD))
        ang = torch.cat([ang, ang], -1)
        return {"h": bf(B, T, c["hidden"]), "g": (1 + 0.1 * _randn(g, c["hidden"])).to(torch.bfloat16),
                "q": bf(B, T, c["heads"], HEAD), "gq": (1 + 0.1 * _randn(g, HEAD)).to(torch.bfloat16),
                "cos": ang.cos().to(torch.bfloat16), "sin": ang.sin().to(torch.bfloat16),
                "a": bf(B, T, c["inter"]), "b": bf(B, T, c["inter"])}
    if kind == "statistics":
        s = _channels(g, c["n"])
        xq = _activations(g, c["N"], c["n"], s)
        xr = (xq.float() + 0.05 * _randn(g, c["N"], c["n"]) * s).to(torch.bfloat16) if c["cross"] else None
        return {"xq": xq, "xr": xr, "w": _digit_weights(g, c["N"]) if c["weighted"] else None}
    if kind in ("factor", "rotation"):
        return {"H": _statistics(g, c["n"])}
    if kind == "qep":
        H = _statistics(g, c["n"])
        return {"H": H, "D": 0.02 * H + 0.01 * H.diagonal().mean() * _randn(g, c["n"], c["n"], dtype=torch.float64)
                / math.sqrt(c["n"]), "W": (0.015 * _randn(g, c["m"], c["n"])).to(torch.bfloat16)}
    if kind == "sweep":
        return {"H": _statistics(g, c["n"]), "W": 0.02 * _randn(g, c["m"], c["n"], dtype=torch.float64)}
    if kind == "lloyd":
        return {"H": _statistics(g, c["n"]), "X": _randn(g, c["m"], c["n"], dtype=torch.float64)}
    if kind == "viterbi":
        return {"X": _randn(g, c["B"], c["T"], dtype=torch.float64)}
    ref = (3.0 * _randn(g, c["T"], c["V"])).to(torch.bfloat16 if c["dtype"] == "bf16" else torch.float32)
    q = (ref.float() + 0.3 * _randn(g, c["T"], c["V"])).to(ref.dtype)
    return {"ref": ref, "q": q}


def prepare(case: dict, seed: int) -> dict:
    st = {"case": case, "seed": int(seed) % 100003} | _inputs(case, seed)
    if case["kind"] == "sweep":
        # the stage's plan, tables and factor, which the layer loop has made before the sweep
        st["groups"] = _row_groups(seed, case["m"], case["bits"])
        st["tables"] = {k: _table(case["L"], k) for k in sorted({g["bits"] for g in st["groups"]})}
        st["factor"] = quantize.stage_factor(st["H"], st["seed"])
    elif case["kind"] == "lloyd":
        st["U"] = ldlq_gpu.ldlq_factor(st["H"])
        n = case["levels"]
        st["levels"] = torch.special.ndtri((torch.arange(n, dtype=torch.float64) + 0.5) / n).to(DEV)
    elif case["kind"] == "viterbi":
        st["values"] = _table(case["L"], case["k"])
    return st


# ----------------------------------------------------------------------------- one pass


def run(st: dict):
    c = st["case"]
    kind = c["kind"]
    if kind == "attention":
        return engine.attention_causal(st["q"], st["k"], st["v"], 1.0 / math.sqrt(HEAD))
    if kind == "pointwise":
        return (engine.rms_norm(st["h"], st["g"], 1e-6, engine.row_pad(c["hidden"])),
                engine.rms_norm_rope(st["q"], st["gq"], 1e-6, st["cos"], st["sin"]),
                engine.swiglu(st["a"], st["b"]))
    if kind == "statistics":
        H, D = quantize.stage_statistics([st["xq"]], None if st["w"] is None else [st["w"]],
                                         None if st["xr"] is None else [st["xr"]])
        return H if D is None else (H, D)
    if kind == "factor":
        env = Environment(st["H"])
        return env.H, env.U, env.dead
    if kind == "rotation":
        return engine.rotate_hessian(st["H"], st["seed"])
    if kind == "qep":
        return quantize.qep_targets(st["H"], st["D"], 0.5, {"w": st["W"]})["w"]
    if kind == "sweep":
        return quantize.quantize_stage_row_groups({"w": st["W"]}, {"w": st["groups"]}, st["H"], st["seed"], L=c["L"],
                                                  tables=st["tables"], factor=st["factor"])["w"]
    if kind == "lloyd":
        return ldlq_gpu.ldlq_round(st["X"], st["U"], st["levels"])
    if kind == "viterbi":
        return codes.viterbi(st["X"], st["values"], c["L"], c["k"])
    return compiler.kl_per_token(st["ref"], st["q"])


# ----------------------------------------------------------------------------- work


def _kronecker_adds(n: int) -> float:
    """Additions per row of the rotation: the power-of-two factor as a fast transform, the other as its products."""
    p2 = n & -n
    p = n // p2
    if p == 1:
        return n * math.log2(n)
    q = p
    while not (_is_prime(q - 1) and q % 4 == 0):
        q *= 2
    return n * (math.log2(n // q) + q)


def work(case: dict) -> dict:
    c, kind = case, case["kind"]
    if kind == "attention":
        B, T, H, kv = c["B"], c["T"], c["heads"], c["kv"]
        return {"bytes": 2.0 * B * T * HEAD * (2 * H + 2 * kv), "flops": 4.0 * B * H * HEAD * T * (T + 1) / 2}
    if kind == "pointwise":
        rows = c["B"] * c["T"]
        el = 2 * c["hidden"] + 2 * c["heads"] * HEAD + 3 * c["inter"]
        return {"bytes": 2.0 * rows * el + 4.0 * c["T"] * HEAD, "flops": 8.0 * rows * el}
    if kind == "statistics":
        N, n = c["N"], c["n"]
        by = 2.0 * N * n * (2 if c["cross"] else 1) + (4.0 * N if c["weighted"] else 0)
        return {"bytes": by + 8.0 * n * n * (2 if c["cross"] else 1),
                "flops": float(N) * n * (n + 1) + (2.0 * N * n * n if c["cross"] else 0.0)}
    if kind == "factor":
        return {"bytes": 24.0 * c["n"] ** 2, "flops": 2.0 * c["n"] ** 3 / 3}
    if kind == "rotation":
        return {"bytes": 16.0 * c["n"] ** 2, "flops": 2.0 * c["n"] * _kronecker_adds(c["n"])}
    if kind == "qep":
        n, m = float(c["n"]), float(c["m"])
        return {"bytes": 16.0 * n * n + 10.0 * m * n,
                "flops": 2.0 * n ** 3 / 3 + min(4.0 * m * n * n, 2.0 * n ** 3 + 2.0 * m * n * n)}
    if kind == "sweep":
        n, m, L = c["n"], c["m"], c["L"]
        bits = [int(b) for b in c["bits"]]
        ops = sum(sum(engine.trellis_block_ops(n, L, b)) for b in bits) / len(bits) * m
        return {"bytes": 12.0 * m * n + 8.0 * n * n + 8.0 * m, "flops": ops + float(m) * n * n}
    if kind == "lloyd":
        return {"bytes": 16.0 * c["m"] * c["n"] + 8.0 * c["n"] ** 2, "flops": float(c["m"]) * c["n"] ** 2}
    if kind == "viterbi":
        return {"bytes": 16.0 * c["B"] * c["T"] + 8.0 * (1 << c["L"]),
                "flops": float(c["B"]) * c["T"] * engine.viterbi_ops_per_row_step(c["L"], c["k"])}
    el = c["T"] * c["V"]
    return {"bytes": 2.0 * el * (2 if c["dtype"] == "bf16" else 4) + 4.0 * c["T"], "flops": 10.0 * el}


# ----------------------------------------------------------------------------- correctness


def tolerance(case: dict):
    kind = case["kind"]
    if kind in ("attention", "pointwise"):
        return {"rel": 1e-2, "max": 0.1}  # bf16 results (one rounding is 2e-3 of a value)
    if kind == "statistics":
        return {"rel": 2e-5, "max": 1e-3}  # float32 sums over the tokens
    if kind == "factor":
        return {"rel": 1e-11, "max": 1e-8}  # float64; the conditioning of the damped moment
    if kind == "rotation":
        return {"rel": 1e-13, "max": 1e-11}
    if kind == "qep":
        return {"rel": 1e-12, "max": 1e-9}
    if kind == "sweep":
        # states, and float64 row scales; a state differs only where a float32 cost ties to within float64 rounding
        return {"rel": 1e-13, "max": 1e-12, "differ": 2e-4}
    if kind in ("lloyd", "viterbi"):
        return "exact"
    return {"rel": 1e-5, "max": 1e-3}  # float32 sums over the vocabulary


def _is_prime(q: int) -> bool:
    return q > 1 and all(q % d for d in range(2, math.isqrt(q) + 1))


def _dense_rotation(n: int, seed: int) -> torch.Tensor:
    """R = (A kron B) diag(s) / sqrt(n): A the largest Sylvester factor whose cofactor is 1, 2 or a Paley order."""
    a = n & -n
    while True:
        p = n // a
        if p in (1, 2) or (p % 4 == 0 and _is_prime(p - 1)):
            break
        a //= 2
    B = torch.ones(1, 1, dtype=torch.float64)
    if p > 2:
        q = p - 1
        squares = {(x * x) % q for x in range(1, q)}
        B = torch.ones(p, p, dtype=torch.float64)
        for i in range(q):
            B[i + 1, 0] = -1.0
            for j in range(q):
                d = (j - i) % q
                B[i + 1, j + 1] = 1.0 if d == 0 or d in squares else -1.0
    elif p == 2:
        a *= 2
    S = torch.ones(1, 1, dtype=torch.float64)
    pair = torch.tensor([[1.0, 1.0], [1.0, -1.0]], dtype=torch.float64)
    while S.shape[0] < a:
        S = torch.kron(S, pair)
    u = torch.rand(n, generator=torch.Generator().manual_seed(int(seed)), dtype=torch.float64)
    return (torch.kron(S, B) / math.sqrt(n) * torch.where(u < 0.5, -1.0, 1.0)[None, :]).to(DEV)


def _norm(x: torch.Tensor, g: torch.Tensor) -> torch.Tensor:
    x = x.double()
    return x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + 1e-6) * g.double()


def exact(case: dict, seed: int):
    c, kind = case, case["kind"]
    s = _inputs(case, seed)
    if kind == "attention":
        B, H, T, D = s["q"].shape
        out = torch.empty(B, T, H, D, dtype=torch.float64, device=DEV).transpose(1, 2)
        mask = torch.ones(T, T, dtype=torch.bool, device=DEV).triu(1)
        for b in range(B):
            for h in range(H):
                kh = h // (H // c["kv"])
                P = s["q"][b, h].double() @ s["k"][b, kh].double().T.contiguous() / math.sqrt(D)
                out[b, h] = P.masked_fill_(mask, -math.inf).softmax(-1) @ s["v"][b, kh].double()
        return out
    if kind == "pointwise":
        y = _norm(s["q"], s["gq"])
        rot = torch.cat([-y[..., HEAD // 2 :], y[..., : HEAD // 2]], -1)
        q = y * s["cos"].double()[None, :, None, :] + rot * s["sin"].double()[None, :, None, :]
        a = s["a"].double()
        return _norm(s["h"], s["g"]), q, a * torch.sigmoid(a) * s["b"].double()
    if kind == "statistics":
        xq = s["xq"].double()
        wx = xq if s["w"] is None else xq * s["w"].double()[:, None]
        H = (wx.T @ xq) / c["N"]
        return H if s["xr"] is None else (H, (s["xr"].double().T @ wx) / c["N"])
    if kind == "factor":
        H = s["H"]
        H = H + 0.01 * H.diagonal().mean() * torch.eye(c["n"], dtype=torch.float64, device=DEV)
        # the upper U with U^T U = H^-1, through the flipped matrix's factor: H = V V^T, V upper, U = V^-1
        V = torch.linalg.cholesky(H.flip(0, 1).cpu()).flip(0, 1).contiguous()
        U = torch.linalg.solve_triangular(V, torch.eye(c["n"], dtype=torch.float64), upper=True)
        return H, U.to(DEV), None
    if kind == "rotation":
        R = _dense_rotation(c["n"], int(seed) % 100003)
        return R @ s["H"] @ R.T
    if kind == "qep":
        H = s["H"] + quantize.LAM * s["H"].diagonal().mean() * torch.eye(c["n"], dtype=torch.float64, device=DEV)
        W = s["W"].double()
        Y = torch.linalg.solve(H.cpu(), (W @ s["D"]).T.contiguous().cpu()).T
        return W + 0.5 * Y.to(DEV)
    if kind == "sweep":
        return None, s["W"].pow(2).mean(1).sqrt().clamp_min(1e-12)  # the rotation keeps a row's RMS
    if kind in ("lloyd", "viterbi"):
        return None
    out = torch.empty(c["T"], dtype=torch.float64, device=DEV)
    for t in range(0, c["T"], 256):
        r = s["ref"][t : t + 256].double().log_softmax(-1)
        out[t : t + 256] = (r.exp() * (r - s["q"][t : t + 256].double().log_softmax(-1))).sum(-1)
    return out
