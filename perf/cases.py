"""The work this library is measured on: the five MoE ops through their public
entry points, over the sizes a serving program gives them.

A case is a dict of plain values with an ``op``:

* ``int4``    ``fused_moe_int4_w4a16`` (one projection of an INT4 MoE layer)
* ``mxfp4``   ``fused_moe_mxfp4`` (a whole MXFP4 expert MLP)
* ``align``   ``moe_align_block_size``
* ``reduce``  ``moe_sum_reduce``
* ``router``  ``topk_softmax``

``listed()`` names the fixed cases, ``draw(rng)`` gives further ones of the same
ranges, ``prepare`` makes a case's inputs on the GPU, ``run`` is one call,
``exact`` the same result in 64 bits with torch alone.
"""
from __future__ import annotations

import math

import torch

import xkernels_amd as xk

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
SIZES = {"bf16": 2, "fp16": 2, "fp32": 4}

# INT4 projections (E experts, N rows, K columns, top_k): the gate/up and the down
# projection of a 384-expert model's expert-parallel shard, the small
# configuration, and one whose K and N are not multiples of 128.
INT4_SHAPES = [(48, 4096, 7168, 8), (48, 7168, 2048, 8), (8, 1024, 2048, 2), (48, 2880, 2880, 4)]
# MXFP4 expert MLPs (E, hidden, ispp, top_k); the last one's sizes are not
# multiples of 128.
MXFP4_SHAPES = [(256, 4096, 512, 6), (64, 2048, 1408, 8), (32, 2880, 2880, 4)]
E2M1 = (0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0, -0.0, -0.5, -1.0, -1.5, -2.0, -3.0, -4.0, -6.0)


def int4(M, shape=0, dtype="bf16", group=32, routing="uniform", experts=0, workspace=True):
    """``experts``: 0, or the model's expert count when this GPU holds the first E
    of them and gets the whole batch's routing with an expert map."""
    E, N, K, top_k = INT4_SHAPES[shape]
    return {"op": "int4", "M": M, "E": E, "N": N, "K": K, "top_k": top_k, "dtype": dtype, "group": group,
            "routing": routing, "experts": experts, "workspace": workspace}


def mxfp4(M, shape=0, bias=False, routing="uniform", workspace=True):
    E, hidden, ispp, top_k = MXFP4_SHAPES[shape]
    return {"op": "mxfp4", "M": M, "E": E, "hidden": hidden, "ispp": ispp, "top_k": top_k, "bias": bias,
            "routing": routing, "workspace": workspace}


def align(M, E, top_k, block, routing, truncate):
    return {"op": "align", "M": M, "E": E, "top_k": top_k, "block": block, "routing": routing,
            "truncate": truncate}


def reduce_(M, top_k, H, dtype, weights, scaling):
    return {"op": "reduce", "M": M, "top_k": top_k, "H": H, "dtype": dtype, "weights": weights,
            "scaling": scaling}


def router(M, E, top_k, dtype, renormalize):
    return {"op": "router", "M": M, "E": E, "top_k": top_k, "dtype": dtype, "renormalize": renormalize}


def listed() -> list[dict]:
    return [
        # the router of a 4096-token prefill batch
        {"name": "router-m4096", **router(4096, 256, 8, "bf16", True)},
        # sorting a large prefill batch's slots by expert, without a host sync
        {"name": "align-m16384", **align(16384, 48, 8, 16, "zipf", False)},
        # combining a prefill batch's expert outputs
        {"name": "reduce-m8192", **reduce_(8192, 8, 7168, "bf16", "fp32", 1.0)},
        # one user's decode step: eight experts' gate/up weights for one token
        {"name": "int4-gateup-m1", **int4(1)},
        # a decode batch of 64 users: every expert's gate/up weights
        {"name": "int4-gateup-m64", **int4(64)},
        # a small decode batch's down projection
        {"name": "int4-down-m16", **int4(16, shape=1)},
        # a large decode batch, or a prompt's last chunk: about 42 rows per expert
        {"name": "int4-gateup-m250", **int4(250)},
        # an expert-parallel rank's share of a large decode batch (48 of 384 experts)
        {"name": "int4-down-ep-m777", **int4(777, shape=1, experts=384)},
        # a prefill batch with skewed expert popularity
        {"name": "int4-gateup-m4096", **int4(4096, routing="zipf", workspace=False)},
        # one user's decode step through an MXFP4 expert MLP
        {"name": "mxfp4-m1", **mxfp4(1)},
        # a decode batch of 48 users
        {"name": "mxfp4-m48", **mxfp4(48)},
        # a prefill batch
        {"name": "mxfp4-m4096", **mxfp4(4096, workspace=False)},
    ]


def _log(rng, lo, hi) -> int:
    """A whole number spread evenly over the logarithm of [lo, hi]."""
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng) -> dict:
    op = rng.choice(["int4"] * 4 + ["mxfp4"] * 3 + ["align", "reduce", "router"])
    routing = rng.choice(["uniform", "zipf"])
    if op == "int4":
        shape = rng.choice([0, 0, 1, 1, 2, 3])
        if rng.random() < 0.15:  # fp32 activations: decode batches
            return int4(_log(rng, 1, 64), shape, "fp32", routing=routing)
        # groups of 64 and 128 where K has them
        group = rng.choice([32, 32, 32, 64, 128]) if INT4_SHAPES[shape][2] % 128 == 0 else 32
        experts = rng.choice([0, 0, 384]) if shape < 2 else 0
        M = _log(rng, 1, 512 if shape == 3 else 4096)
        return int4(M, shape, "bf16", group, routing, experts, workspace=rng.random() < 0.7)
    if op == "mxfp4":
        shape = rng.choice([0, 0, 1, 2])
        return mxfp4(_log(rng, 1, [4096, 2048, 512][shape]), shape, rng.random() < 0.5, routing,
                     workspace=rng.random() < 0.7)
    if op == "align":
        return align(_log(rng, 1, 16384), rng.choice([8, 48, 64, 256, 384]), rng.choice([1, 2, 4, 6, 8]),
                     rng.choice([16, 32, 64, 128]), routing, rng.random() < 0.3)
    if op == "reduce":
        dtype = rng.choice(["bf16", "bf16", "fp32"])
        return reduce_(_log(rng, 1, 8192 if dtype == "bf16" else 4096), rng.choice([1, 2, 4, 6, 8]),
                       rng.choice([2048, 2880, 4096, 7168]), dtype, rng.choice(["fp32", "bf16", "none"]),
                       rng.choice([1.0, 2.5]))
    E = rng.choice([8, 48, 64, 128, 256, 384])
    return router(_log(rng, 1, 16384), E, rng.choice([1, 2, 4, 6, 8]), rng.choice(["bf16", "fp16", "fp32"]),
                  rng.random() < 0.7)


# ------------------------------------------------------------------- inputs ---

def _routing(c, n, g):
    """``top_k`` distinct experts of ``n`` per token: uniform, or popularity
    falling like 1 / rank^1.2 with the ranks dealt out at random; softmax weights."""
    M, k = c["M"], c["top_k"]
    # the top_k largest of log-popularity + Gumbel noise: draws without replacement
    noise = -torch.log(-torch.log(torch.rand(M, n, generator=g, device="cuda").clamp_(1e-7, 1 - 1e-7)))
    if c["routing"] == "zipf":
        rank = torch.randperm(n, generator=g, device="cuda") + 1
        noise = noise - 1.2 * torch.log(rank.float())
    ids = torch.topk(noise, k, dim=1).indices.to(torch.int32)
    w = torch.softmax(torch.randn(M, k, generator=g, device="cuda"), -1)
    return ids, w


def _bytes(shape, g, lo=0, hi=256):
    return torch.randint(lo, hi, shape, generator=g, device="cuda", dtype=torch.uint8)


def prepare(c, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    op, M = c["op"], c["M"]
    s = {"case": c}
    if op == "int4":
        E, N, K, dt = c["E"], c["N"], c["K"], DTYPES[c["dtype"]]
        s["A"] = torch.randn(M, K, generator=g, device="cuda").to(dt)
        s["packed"] = torch.randint(-2**31, 2**31, (E, N, K // 8), generator=g, device="cuda", dtype=torch.int32)
        s["scale"] = (torch.rand(E, N, K // c["group"], generator=g, device="cuda") * 0.015 + 0.005).to(torch.bfloat16)
        s["ids"], s["w"] = _routing(c, c["experts"] or E, g)
        s["map"] = None
        if c["experts"]:
            s["map"] = torch.full((c["experts"],), -1, dtype=torch.int32, device="cuda")
            s["map"][:E] = torch.arange(E, dtype=torch.int32, device="cuda")
        s["ws"] = (xk.MoeInt4Workspace.allocate(M, c["top_k"], N, dtype=dt, device="cuda", num_experts=E, K=K)
                   if c["workspace"] else None)
    elif op == "mxfp4":
        E, h, i = c["E"], c["hidden"], c["ispp"]
        s["A"] = torch.randn(M, h, generator=g, device="cuda").to(torch.bfloat16)
        s["w13"], s["s13"] = _bytes((E, 2 * i, h // 2), g), _bytes((E, 2 * i, h // 32), g, 119, 128)
        s["w2"], s["s2"] = _bytes((E, h, i // 2), g), _bytes((E, h, i // 32), g, 119, 128)
        s["b13"] = s["b2"] = None
        if c["bias"]:
            s["b13"] = (torch.rand(E, 2 * i, generator=g, device="cuda") * 0.2 - 0.1).to(torch.bfloat16)
            s["b2"] = (torch.rand(E, h, generator=g, device="cuda") * 0.2 - 0.1).to(torch.bfloat16)
        s["ids"], s["w"] = _routing(c, E, g)
        s["ws"] = (xk.MoeMxfp4Workspace.allocate(M, c["top_k"], E, 16, i, h, dtype=torch.bfloat16, device="cuda")
                   if c["workspace"] else None)
    elif op == "align":
        s["ids"], _ = _routing(c, c["E"], g)
        s["ws"] = xk.MoeAlignWorkspace.allocate(M, c["top_k"], c["E"], c["block"], device="cuda")
    elif op == "reduce":
        s["y"] = torch.randn(M, c["top_k"], c["H"], generator=g, device="cuda", dtype=DTYPES[c["dtype"]])
        s["w"] = None
        if c["weights"] != "none":
            s["w"] = torch.softmax(torch.randn(M, c["top_k"], generator=g, device="cuda"), -1).to(DTYPES[c["weights"]])
    else:
        s["logits"] = torch.randn(M, c["E"], generator=g, device="cuda").to(DTYPES[c["dtype"]])
    return s


def run(s):
    c = s["case"]
    op = c["op"]
    if op == "int4":
        return xk.fused_moe_int4_w4a16(s["A"], s["packed"], s["scale"], s["ids"], s["w"], group_size=c["group"],
                                       expert_map=s["map"], workspace=s["ws"])
    if op == "mxfp4":
        return xk.fused_moe_mxfp4(s["A"], s["w13"], s["s13"], s["w2"], s["s2"], s["ids"], s["w"], b13=s["b13"],
                                  b2=s["b2"], workspace=s["ws"])
    if op == "align":
        return xk.moe_align_block_size(s["ids"], c["block"], c["E"], truncate=c["truncate"], workspace=s["ws"])
    if op == "reduce":
        return xk.moe_sum_reduce(s["y"], s["w"], routed_scaling_factor=c["scaling"])
    return xk.topk_softmax(s["logits"], c["top_k"], renormalize=c["renormalize"])


# ---------------------------------------------------------------- work, tolerance ---

def _active(c) -> float:
    """Experts expected to get at least one of the batch's slots (uniform routing)."""
    return c["E"] * (1.0 - (1.0 - c["top_k"] / (c.get("experts") or c["E"])) ** c["M"])


def work(c) -> dict:
    op, M = c["op"], c["M"]
    if op == "int4":
        E, N, K = c["E"], c["N"], c["K"]
        slots = M * c["top_k"] * (E / c["experts"] if c["experts"] else 1.0)
        weights = _active(c) * (N * K / 2 + N * (K // c["group"]) * 2)
        return {"bytes": weights + M * (K + N) * SIZES[c["dtype"]] + M * c["top_k"] * 8,
                "flops": 2.0 * slots * N * K}
    if op == "mxfp4":
        h, i = c["hidden"], c["ispp"]
        weights = _active(c) * 3 * h * i * (0.5 + 1 / 32)
        return {"bytes": weights + M * h * 4 + M * c["top_k"] * 8, "flops": 6.0 * M * c["top_k"] * h * i}
    if op == "align":
        numel = M * c["top_k"]
        most = numel + (c["E"] + 1) * (c["block"] - 1)
        return {"bytes": numel * 4 + most * 4 + most // c["block"] * 4, "flops": 0}
    if op == "reduce":
        size, wsize = SIZES[c["dtype"]], SIZES.get(c["weights"], 0)
        return {"bytes": M * c["H"] * (c["top_k"] + 1) * size + M * c["top_k"] * wsize,
                "flops": 2.0 * M * c["top_k"] * c["H"]}
    return {"bytes": M * c["E"] * SIZES[c["dtype"]] + M * c["top_k"] * 8, "flops": 4.0 * M * c["E"]}


def tolerance(c):
    """About four times the distance from ``exact`` (measured): the output's own
    rounding for one product or sum in bf16, plus the three bf16 roundings inside
    the MXFP4 MLP; fp32 sums and, with fp32 activations, their bf16 triple product."""
    op = c["op"]
    if op == "align":
        return "exact"
    if op == "mxfp4":
        return {"rel": 1e-2, "max": 0.1}
    if op == "router":
        return {"rel": 3e-7, "max": 3e-6, "differ": 1e-4}
    if c["dtype"] == "bf16":
        return {"rel": 7e-3, "max": 2e-2}
    return {"rel": 1.5e-5, "max": 2e-4} if op == "int4" else {"rel": 1e-6, "max": 1e-5}


# ------------------------------------------------------------------- 64 bits ---

def _unpack(b, values):
    """[rows, bytes] uint8 -> [rows, 2 * bytes] of ``values[nibble]``, low nibble first."""
    b = b.long()
    return torch.stack((values[b & 15], values[b >> 4]), -1).reshape(b.shape[0], -1)


def _int4_exact(s):
    c, A = s["case"], s["A"].double()
    out = torch.zeros(c["M"], c["N"], dtype=torch.float64, device="cuda")
    values = torch.arange(16, device="cuda", dtype=torch.float64) - 8
    for e in range(c["E"]):  # expert maps here keep the first E experts
        m, j = torch.nonzero(s["ids"] == e, as_tuple=True)
        if m.numel() == 0:
            continue
        W = _unpack(s["packed"][e].view(torch.uint8), values)
        W = (W.view(c["N"], -1, c["group"]) * s["scale"][e].double().unsqueeze(-1)).view(c["N"], c["K"])
        if c["dtype"] == "bf16":  # the op rounds a weight to the activations' type
            W = W.to(torch.bfloat16).double()
        out.index_add_(0, m, A[m] @ W.t() * s["w"][m, j].double().unsqueeze(-1))
    return out


def _mxfp4_exact(s, limit=10.0):
    c, A = s["case"], s["A"].double()
    i = c["ispp"]
    out = torch.zeros(c["M"], c["hidden"], dtype=torch.float64, device="cuda")
    values = torch.tensor(E2M1, device="cuda", dtype=torch.float64)

    def weight(q, sc, e):
        W = _unpack(q[e], values)
        return (W.view(W.shape[0], -1, 32) * torch.exp2(sc[e].double() - 127).unsqueeze(-1)).view(W.shape)

    for e in range(c["E"]):
        m, j = torch.nonzero(s["ids"] == e, as_tuple=True)
        if m.numel() == 0:
            continue
        gu = A[m] @ weight(s["w13"], s["s13"], e).t()
        if s["b13"] is not None:
            gu = gu + s["b13"][e].double()
        gate, up = gu[:, :i].clamp(max=limit), gu[:, i:].clamp(-limit, limit)
        down = (torch.nn.functional.silu(gate) * up) @ weight(s["w2"], s["s2"], e).t()
        if s["b2"] is not None:
            down = down + s["b2"][e].double()
        out.index_add_(0, m, down * s["w"][m, j].double().unsqueeze(-1))
    return out


def exact(c, seed):
    if c["op"] == "align":
        return None
    s = prepare({**c, "workspace": False}, seed)
    if c["op"] == "int4":
        return _int4_exact(s)
    if c["op"] == "mxfp4":
        return _mxfp4_exact(s)
    if c["op"] == "reduce":
        out = torch.empty(c["M"], c["H"], dtype=torch.float64, device="cuda")
        for m in range(0, c["M"], 1024):  # a part at a time: the whole in 64 bits is large
            y = s["y"][m:m + 1024].double()
            if s["w"] is not None:
                y = y * s["w"][m:m + 1024].double().unsqueeze(-1)
            out[m:m + 1024] = y.sum(1) * c["scaling"]
        return out
    p = torch.softmax(s["logits"].double(), -1)
    w = torch.topk(p, c["top_k"], dim=1).values
    if c["renormalize"]:
        w = w / w.sum(1, keepdim=True)
    return w, None
