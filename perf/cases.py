"""The performance cases: what a program on this backend has it do.

Each case goes through the entry points such a program calls: a compiled program
(``tempest_hip.compile`` and a call of what it returns, which copies the results and reads
the numbers), or a built launch run on arrays the program keeps.  ``listed`` names the cases,
``draw`` makes more of the same ranges, ``prepare`` makes a case's inputs and handles, ``run``
is one pass, ``exact`` the same results in float64 by plain torch.

Arrays are the library's column-major layouts, so a torch tensor holding one has the reversed
shape: attention's (d, heads, positions, batch) is a (B, S, H, D) tensor here.
"""
from __future__ import annotations

import functools
import math
import sys

import torch

sys.path[:0] = ["tempest.jl_amd"]  # the package's folder, from the repository's root

import tempest_hip as th  # noqa: E402
import tempest_hip.launch as L  # noqa: E402

F32, BF16, F64 = torch.float32, torch.bfloat16, torch.float64


@functools.lru_cache(maxsize=None)
def _target() -> th.HIPTarget:
    return th.HIPTarget()


# ---- the cases -------------------------------------------------------------------------

def listed() -> list[dict]:
    return [
        # The smallest program, a dense tanh layer's loss and gradient, as its caller waits for
        # it: one kernel, so dispatch, the results' copy and the loss's read are the time.
        {"name": "tanh_call", "kind": "tanh", "d": 32, "h": 64, "c": 16},
        # Softmax with its gradient over a large activation: rows resident, HBM-bound.
        {"name": "softmax_grad_large", "kind": "rows", "op": "softmax", "floor": False, "rows": 32768, "n": 8192},
        # LayerNorm with its gradient as the planner's own groups (generated kernels), at a
        # ragged row length that no wide load divides.
        {"name": "layernorm_grad_generated", "kind": "rows", "op": "layernorm", "floor": True, "rows": 6000, "n": 3001},
        # A two-layer GELU MLP's training step, bf16: the largest products...
        {"name": "mlp_grad_large", "kind": "mlp", "batch": 4096, "d_in": 4096, "hidden": 16384, "d_out": 4096},
        # ... and at the width and batch of a small transformer's block.
        {"name": "mlp_grad_small", "kind": "mlp", "batch": 1024, "d_in": 768, "hidden": 3072, "d_out": 768},
        # Causal attention's training step, bf16, long sequences, compiled.
        {"name": "attention_grad_d128", "kind": "attention", "B": 8, "H": 16, "KV": 16, "S": 4096, "D": 128,
         "causal": True, "f32": False, "grad": True},
        # The same for a small model: 64 features, grouped heads, a ragged length.
        {"name": "attention_grad_d64", "kind": "attention", "B": 4, "H": 12, "KV": 4, "S": 1023, "D": 64,
         "causal": True, "f32": False, "grad": True},
        # fp32 attention in full precision, the default of fp32 programs.
        {"name": "attention_grad_f32", "kind": "attention", "B": 2, "H": 8, "KV": 8, "S": 1024, "D": 64,
         "causal": True, "f32": True, "grad": True},
        # Decode: one query a sequence over a cache whose lengths the device holds, grouped heads.
        {"name": "attention_decode", "kind": "decode", "B": 16, "H": 32, "KV": 8, "cache": 4096, "D": 128},
        # Training on documents packed in sequences (a first key per query).
        {"name": "attention_packed", "kind": "packed", "B": 2, "H": 12, "KV": 12, "S": 2048, "D": 64, "docs": 8},
        # A chunked gated DeltaNet layer's training step.
        {"name": "deltanet_grad", "kind": "deltanet", "B": 4, "H": 16, "T": 8192},
        # A product of fp32 factors in full precision, sizes no tile divides.
        {"name": "product_f32", "kind": "product", "m": 2000, "n": 1500, "k": 1030, "dtype": "f32"},
    ]


def _log(rng, lo: int, hi: int) -> int:
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng) -> dict:
    kind = rng.choice(["tanh", "rows", "rows", "mlp", "mlp", "attention", "attention", "attention_f32", "decode",
                       "decode", "packed", "packed", "deltanet", "product", "product"])
    if kind == "tanh":
        return {"kind": kind, "d": rng.randint(8, 48), "h": rng.randint(8, 96), "c": rng.randint(1, 48)}
    if kind == "rows":
        n = _log(rng, 64, 16384)
        rows = _log(rng, 256, min(32768, (1 << 28) // n))
        return {"kind": kind, "op": rng.choice(["softmax", "layernorm"]), "floor": rng.random() < 0.4, "rows": rows,
                "n": n}
    if kind == "mlp":  # the fused products take sizes in 8s
        d = 8 * _log(rng, 32, 512)
        return {"kind": kind, "batch": 8 * _log(rng, 16, 512), "d_in": d, "hidden": d * rng.choice([2, 4]),
                "d_out": rng.choice([d, 8 * _log(rng, 32, 512)])}
    if kind in ("attention", "attention_f32"):
        f32 = kind == "attention_f32"
        kv, group = rng.choice([2, 4, 8]), rng.choice([1, 1, 2, 4])
        d, s = rng.choice([64, 128]), _log(rng, 128, 2048 if f32 else 4096)
        s = rng.choice([s, (s + 127) // 128 * 128])  # ragged, or padded as a loader would
        most = (1 << 16) if f32 else (1 << 19)  # batch x heads x positions
        b = max(1, min(8, most // (kv * group * s)))
        return {"kind": "attention", "B": rng.randint(1, b), "H": kv * group, "KV": kv, "S": s, "D": d,
                "causal": rng.random() < 0.75, "f32": f32, "grad": rng.random() < 0.7}
    if kind == "decode":
        kv, d, cache = rng.choice([1, 2, 4, 8]), rng.choice([64, 128]), _log(rng, 200, 16384)
        b = max(1, min(64, (1 << 26) // (kv * d * cache)))  # the cache's elements
        return {"kind": kind, "B": rng.randint(1, b), "H": kv * rng.choice([1, 2, 4, 8]), "KV": kv, "cache": cache,
                "D": d}
    if kind == "packed":
        kv, group, s = rng.choice([2, 4, 8]), rng.choice([1, 1, 2]), _log(rng, 256, 4096)
        b = max(1, min(4, (1 << 16) // (kv * group * s)))
        return {"kind": kind, "B": rng.randint(1, b), "H": kv * group, "KV": kv, "S": s, "D": rng.choice([64, 128]),
                "docs": rng.randint(2, 24)}
    if kind == "deltanet":
        return {"kind": kind, "B": rng.randint(1, 4), "H": rng.choice([4, 8, 12, 16]), "T": 64 * _log(rng, 4, 128)}
    m, n, k = _log(rng, 64, 4096), _log(rng, 64, 4096), _log(rng, 64, 4096)
    dtype = rng.choice(["f32", "f32", "bf16"])
    if dtype == "bf16":  # leading dimensions in 8s, as a program that uses matrix cores pads them
        m, n, k = (8 * max(8, x // 8) for x in (m, n, k))
    return {"kind": "product", "m": m, "n": n, "k": k, "dtype": dtype}


# ---- inputs ----------------------------------------------------------------------------

def _rng(seed: int):
    gen = torch.Generator(device="cuda").manual_seed(int(seed) % (1 << 62))
    return lambda *shape: torch.randn(*shape, device="cuda", generator=gen)


def _lengths(c: dict, seed: int) -> torch.Tensor:
    """Decode: sequences at every stage of filling the cache, one of them full."""
    gen = torch.Generator().manual_seed(int(seed) % (1 << 62) + 1)
    n = torch.randint(max(1, c["cache"] // 8), c["cache"] + 1, (c["B"],), generator=gen, dtype=torch.int32)
    n[int(torch.randint(0, c["B"], (1,), generator=gen))] = c["cache"]
    return n


def _starts(c: dict, seed: int) -> torch.Tensor:
    """Packed documents: `docs` of random lengths a sequence; each position's 1-based first key."""
    gen = torch.Generator().manual_seed(int(seed) % (1 << 62) + 2)
    out = torch.empty(c["B"], c["S"], dtype=torch.int32)
    for b in range(c["B"]):
        cuts = sorted(set(torch.randint(1, c["S"], (c["docs"] - 1,), generator=gen).tolist()))
        for lo, hi in zip([0] + cuts, cuts + [c["S"]]):
            out[b, lo:hi] = lo + 1
    return out


def _inputs(c: dict, seed: int) -> dict:
    r, kind = _rng(seed), c["kind"]
    if kind == "tanh":
        d, h, n = c["d"], c["h"], c["c"]
        return {"w": r(h, d), "b": r(h) * 0.3, "x": r(n, d) * 0.7}
    if kind == "rows":
        x = r(c["rows"], c["n"])
        return {"x": x, "g": r(c["rows"], c["n"]) + 0.5 * x}  # an upstream gradient that leans with x
    if kind == "mlp":
        di, hid, do = c["d_in"], c["hidden"], c["d_out"]
        return {"W1": (r(di, hid) / di ** 0.5).to(BF16), "b1": (r(hid) / di ** 0.5).to(BF16),
                "W2": (r(hid, do) / hid ** 0.5).to(BF16), "b2": (r(do) / hid ** 0.5).to(BF16),
                "x": r(c["batch"], di).to(BF16)}
    if kind in ("attention", "packed"):
        dt = F32 if c.get("f32") else BF16
        B, S, H, KV, D = c["B"], c["S"], c["H"], c["KV"], c["D"]
        i = {"q": r(B, S, H, D).to(dt), "k": r(B, S, KV, D).to(dt), "v": r(B, S, KV, D).to(dt),
             "dout": r(B, S, H, D).to(dt)}
        if kind == "packed":
            i["starts"] = _starts(c, seed).cuda()
        return i
    if kind == "decode":
        B, n, KV, D = c["B"], c["cache"], c["KV"], c["D"]
        return {"q": r(B, 1, c["H"], D).to(BF16), "k": r(B, n, KV, D).to(BF16), "v": r(B, n, KV, D).to(BF16),
                "lengths": _lengths(c, seed).cuda()}
    if kind == "deltanet":
        B, T, H = c["B"], c["T"], c["H"]
        unit = lambda x: x / x.norm(dim=-1, keepdim=True)  # noqa: E731
        return {"q": unit(r(B, T, H, 128)).to(BF16), "k": unit(r(B, T, H, 128)).to(BF16),
                "v": r(B, T, H, 128).to(BF16), "a": -torch.nn.functional.softplus(r(B, T, H)),
                "beta": torch.sigmoid(r(B, T, H)), "dout": r(B, T, H, 128).to(BF16)}
    dt = F32 if c["dtype"] == "f32" else BF16
    return {"a": r(c["m"], c["k"]).to(dt), "b": r(c["k"], c["n"]).to(dt)}  # A k-contiguous, B n-contiguous


def prepare(case: dict, seed: int) -> dict:
    c, i = case, _inputs(case, seed)
    p = {k: v.data_ptr() for k, v in i.items()}
    kind = c["kind"]
    compiled = {"tanh": lambda: th.programs.tanh_layer(c["d"], c["h"], c["c"]),
                "rows": lambda: getattr(th.programs, {"softmax": "softmax_columns", "layernorm": "layernorm"}[c["op"]]
                                        if not c["floor"] else
                                        {"softmax": "floor_softmax_columns", "layernorm": "floor_layernorm"}[c["op"]])(
                                            c["rows"], c["n"]),
                "mlp": lambda: th.programs.mlp(c["batch"], c["d_in"], c["hidden"], c["d_out"]),
                "deltanet": lambda: th.programs.deltanet(c["B"], c["H"], c["T"])}
    if kind == "attention" and c["D"] == 128 and c["grad"] and not c["f32"]:
        compiled["attention"] = lambda: th.programs.attention(c["B"], c["H"], c["S"], causal=c["causal"],
                                                              kv_heads=c["KV"])
    if kind in compiled:
        args = list(i.values())
        return {"call": th.compile(compiled[kind](), _target(), *args), "args": args}
    _target()
    if kind == "product":
        m, n, k = c["m"], c["n"], c["k"]
        f32 = c["dtype"] == "f32"
        out = torch.empty(n, m, device="cuda", dtype=F32 if f32 else BF16)
        dt = L.F32 if f32 else L.BF16
        launch = L.gemm(m, n, k, p["a"], k, 1, p["b"], n, 1, out.data_ptr(), m, c_dtype=dt, factors=dt)
        return {"launches": [launch], "outputs": [out], "keep": i}
    # attention, packed documents, decode: the forward's launch and, in training, the backward's
    B, S, H, KV, D = c["B"], c.get("S", 1), c["H"], c["KV"], c["D"]
    f32, causal, grad = c.get("f32", False), c.get("causal", kind == "packed"), c.get("grad", kind == "packed")
    extra = {"head_dim": D, "f32": f32, "kv_seq": c.get("cache", S)}
    extra.update({m: p[m] for m in ("starts", "lengths") if m in p})
    o = torch.empty_like(i["q"])
    lse = torch.empty(B, S, H, device="cuda")
    outputs = [o, lse]
    launches = [L.attention_fwd(B, H, KV, S, p["q"], p["k"], p["v"], o.data_ptr(), lse.data_ptr(), causal=causal,
                                **extra)]
    if grad:
        d = [torch.empty_like(i[x]) for x in ("q", "k", "v")]
        outputs += d
        launches.append(L.attention_bwd(B, H, S, p["q"], p["k"], p["v"], o.data_ptr(), lse.data_ptr(), p["dout"],
                                        *(t.data_ptr() for t in d), causal=causal, kv_heads=KV, **extra))
    return {"launches": launches, "outputs": outputs, "keep": i}


def run(state: dict):
    if "call" in state:
        return state["call"](*state["args"])
    for launch in state["launches"]:
        launch()
    return state["outputs"]


# ---- what a pass cannot do without -----------------------------------------------------

def _pairs(c: dict) -> float:
    """(query, key) pairs a head sees, over the batch."""
    if c["kind"] == "packed":
        mean = c["S"] / c["docs"]
        return c["B"] * c["S"] * (2 * mean if c["docs"] > 2 else 1.5 * mean) / 2  # cut at random points
    return c["B"] * c["S"] * ((c["S"] + 1) / 2 if c["causal"] else c["S"])


def work(case: dict) -> dict:
    c, kind = case, case["kind"]
    if kind == "tanh":
        d, h, n = c["d"], c["h"], c["c"]
        return {"bytes": 4 * (2 * d * h + 2 * h + 2 * d * n + 1), "flops": 6 * d * h * n}
    if kind == "rows":
        return {"bytes": 12 * c["rows"] * c["n"], "flops": 12 * c["rows"] * c["n"]}
    if kind == "mlp":
        b, di, hid, do = c["batch"], c["d_in"], c["hidden"], c["d_out"]
        return {"bytes": 2 * (2 * (di * hid + hid + hid * do + do + b * di)), "flops": 6 * b * hid * (di + do)}
    if kind in ("attention", "packed"):
        e = 4 if c.get("f32") else 2
        q, k = c["B"] * c["S"] * c["H"] * c["D"] * e, c["B"] * c["S"] * c["KV"] * c["D"] * e
        grad = c.get("grad", True)
        return {"bytes": (4 * q + 4 * k) if grad else (2 * q + 2 * k),
                "flops": 4 * c["H"] * c["D"] * _pairs(c) * (3.5 if grad else 1)}
    if kind == "decode":
        held = c["B"] * c["cache"] * 9 / 16  # lengths spread evenly over 1/8..1 of the cache
        return {"bytes": 4 * held * c["KV"] * c["D"] + 4 * c["B"] * c["H"] * c["D"],
                "flops": 4 * held * c["H"] * c["D"]}
    if kind == "deltanet":
        t = c["B"] * c["T"] * c["H"]
        return {"bytes": t * (2 * 128 * 8 + 4 * 4), "flops": t * 128 * 128 * 2 * 3 * 3}
    e = 4 if c["dtype"] == "f32" else 2
    m, n, k = c["m"], c["n"], c["k"]
    return {"bytes": e * (m * k + k * n + m * n), "flops": 2 * m * n * k}


def tolerance(case: dict) -> dict:
    """About four times the largest error against ``exact`` over the listed and ninety drawn cases."""
    kind = case["kind"]
    if kind in ("tanh", "rows") or case.get("f32") or case.get("dtype") == "f32":
        return {"rel": 4e-6}   # fp32 throughout: 0.9e-7 (rows) to 1.1e-6 (products 4096 deep)
    if kind == "mlp":
        return {"rel": 1.5e-2}  # bf16 results of stored bf16 values: 3.9e-3
    if kind in ("decode", "product"):
        return {"rel": 7e-3}   # one rounding to bf16: 1.7e-3
    return {"rel": 1e-2}       # attention and its gradients, DeltaNet: 1.7e-3 to 2.5e-3


# ---- the same in float64 ---------------------------------------------------------------

def _rows_exact(c, i):
    dx, loss = torch.empty(c["rows"], c["n"], dtype=F64, device="cuda"), 0.0
    for lo in range(0, c["rows"], 2048):
        x, g = i["x"][lo:lo + 2048].double(), i["g"][lo:lo + 2048].double()
        if c["op"] == "softmax":
            y = torch.softmax(x, dim=1)
            dx[lo:lo + 2048] = y * (g - (y * g).sum(1, keepdim=True))
        else:
            xc = x - x.mean(1, keepdim=True)
            rs = 1.0 / torch.sqrt((xc * xc).mean(1, keepdim=True) + 1e-5)
            y = xc * rs
            dx[lo:lo + 2048] = rs * (g - g.mean(1, keepdim=True) - y * (y * g).mean(1, keepdim=True))
        loss += float((y * g).sum())
    return loss, dx


def _mlp_exact(i):
    W1, b1, W2, b2, x = (i[n].double() for n in ("W1", "b1", "W2", "b2", "x"))
    z = x @ W1 + b1
    u = math.sqrt(2 / math.pi) * (z + 0.044715 * z ** 3)
    t = torch.tanh(u)
    y = 0.5 * z * (1 + t) @ W2 + b2
    dy = 2 * y
    dW2 = (0.5 * z * (1 + t)).t() @ dy
    dz = (dy @ W2.t()) * (0.5 * (1 + t) + 0.5 * z * (1 - t * t) * math.sqrt(2 / math.pi) * (1 + 3 * 0.044715 * z * z))
    return float((y * y).sum()), x.t() @ dz, dz.sum(0), dW2, dy.sum(0), dz @ W1.t()


def _attention_exact(c, i, grad, compiled):
    kind = c["kind"]
    B, H, group, D = c["B"], c["H"], c["H"] // c["KV"], c["D"]
    S, K = i["q"].shape[1], i["k"].shape[1]
    o, lse = torch.empty(B, S, H, D, dtype=F64, device="cuda"), torch.empty(B, S, H, dtype=F64, device="cuda")
    dq = torch.zeros_like(o)
    dk, dv = (torch.zeros(B, K, c["KV"], D, dtype=F64, device="cuda") for _ in range(2))
    keys = torch.arange(K, device="cuda")
    for b in range(B):
        hidden = torch.zeros(S, K, dtype=torch.bool, device="cuda")
        if c.get("causal", kind == "packed"):
            hidden |= keys[None, :] > torch.arange(S, device="cuda")[:, None]
        if kind == "packed":
            hidden |= keys[None, :] < (i["starts"][b].long() - 1)[:, None]
        if kind == "decode":
            hidden |= keys[None, :] >= i["lengths"][b].long()
        for h in range(H):
            q, k, v = i["q"][b, :, h].double(), i["k"][b, :, h // group].double(), i["v"][b, :, h // group].double()
            s = (q @ k.t() / math.sqrt(D)).masked_fill_(hidden, -math.inf)
            lse[b, :, h] = torch.logsumexp(s, 1)
            p = torch.exp(s - lse[b, :, h, None])
            o[b, :, h] = p @ v
            if grad:
                g = i["dout"][b, :, h].double()
                dv[b, :, h // group] += p.t() @ g
                ds = p * (g @ v.t() - (g * o[b, :, h]).sum(1, keepdim=True)) / math.sqrt(D)
                dq[b, :, h] = ds @ k
                dk[b, :, h // group] += ds.t() @ q
    if compiled:
        return [o, dq, dk, dv]
    return [o, lse, dq, dk, dv] if grad else [o, lse]


def _deltanet_exact(c, i):
    """The gated delta rule in chunks of 64, S from zero: U solves (I + A) U = beta (V - e^c K S),
    A the strictly lower part of beta_t e^(c_t - c_j) k_t.k_j, c the chunk's running log-gate;
    (I + A)^-1 as the product of (I + (-A)^(2^j)), A^64 = 0.  Its gradient by autograd."""
    B, T, H, n = c["B"], c["T"], c["H"], 64
    leaves = [i[x].double().requires_grad_() for x in ("q", "k", "v", "a", "beta")]
    q, k, v = (x.transpose(1, 2).reshape(B * H, T, 128) for x in leaves[:3])
    a, beta = (x.transpose(1, 2).reshape(B * H, T) for x in leaves[3:])
    low = torch.tril(torch.ones(n, n, dtype=torch.bool, device="cuda"))
    strict = torch.tril(low, -1)
    eye = torch.eye(n, dtype=F64, device="cuda")
    state, out = torch.zeros(B * H, 128, 128, dtype=F64, device="cuda"), []
    for t in range(0, T, n):
        Q, K, V, b = q[:, t:t + n], k[:, t:t + n], v[:, t:t + n], beta[:, t:t + n, None]
        cum = a[:, t:t + n].cumsum(1)
        gate = torch.exp((cum[:, :, None] - cum[:, None, :]).masked_fill(~low, -math.inf))
        N = -(b * gate * (K @ K.transpose(1, 2))).masked_fill(~strict, 0.0)
        inv = eye + N
        for _ in range(5):
            N = N @ N
            inv = inv + inv @ N
        e = torch.exp(cum)[:, :, None]
        U = inv @ (b * (V - e * (K @ state)))
        out.append(e * (Q @ state) + (gate * (Q @ K.transpose(1, 2))) @ U)
        state = torch.exp(cum[:, -1])[:, None, None] * state + \
            (torch.exp(cum[:, -1:] - cum)[:, :, None] * K).transpose(1, 2) @ U
    o = torch.cat(out, 1).reshape(B, H, T, 128).transpose(1, 2)
    grads = torch.autograd.grad(o, leaves, i["dout"].double())
    return [o.detach().contiguous(), *(g.contiguous() for g in grads)]


def exact(case: dict, seed: int):
    c, i, kind = case, _inputs(case, seed), case["kind"]
    if kind == "tanh":
        w, b, x = (i[n].double() for n in ("w", "b", "x"))
        y = torch.tanh(x @ w.t() + b)
        dz = 2 * y * (1 - y * y)
        return float((y * y).sum()), dz.t() @ x, dz.sum(0), dz @ w
    if kind == "rows":
        return _rows_exact(c, i)
    if kind == "mlp":
        return _mlp_exact(i)
    if kind == "deltanet":
        return _deltanet_exact(c, i)
    if kind == "product":
        return [(i["a"].double() @ i["b"].double()).t().contiguous()]
    compiled = kind == "attention" and c["D"] == 128 and c["grad"] and not c["f32"]
    return _attention_exact(c, i, c.get("grad", kind == "packed"), compiled)
