"""Cases for timing the MoE layer through the entry points that a program calls:
one forward of the op, one forward of the whole block (RMSNorm, op, residual),
one training step (a forward that keeps its values, then the backward of it).

The sizes are those of the repository's benchmark configurations and of the
widths that its tests name (the default expert width round(2.67 D), the example
width D 544), each a piece of real use: see the comments in listed().
"""
from __future__ import annotations

import ctypes
import math
import types

import torch

import mixlab_amd
from mixlab_amd.moe import ffn_dim
from mixlab_amd.op import MoEFeedForward

F32, BF16 = 1, 2               # tensor dtype codes of the C interface
INT8_WEIGHTS, KEEP_FOR_BACKWARD = 16, 32  # create flags
SWIGLU, GEGLU, MLP = 0, 1, 2   # expert kinds
SILU, GELU, RELU, LEAKY_RELU_SQ = 0, 1, 2, 3
EPS, AUX_WEIGHT = 1e-5, 0.01   # the block's norm epsilon and load-balance weight
D_AUX, D_ENTROPY = 0.01, 0.0   # upstream gradients of aux and entropy in a step


def _case(call, dtype, N, D, E, K, F, etype=SWIGLU, act=SILU, zipf=0.0, name=None):
    c = dict(call=call, dtype=dtype, N=N, D=D, E=E, K=K, F=F, etype=etype, act=act, zipf=zipf)
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # one block of the reference's smallest example (moe_tiny: 8 x 128 tokens,
        # D 64, four experts of 128), fp32: launches and latency
        _case("block", "fp32", 1024, 64, 4, 2, 128, name="block_tiny_fp32"),
        # a few sequences decoding, bf16 weights
        _case("forward", "bf16", 8, 1024, 32, 4, 1024, name="decode8_bf16"),
        # 64 sequences decoding on int8 weights (benchmark configuration C5)
        _case("forward", "int8", 64, 2048, 64, 8, 1408, name="decode64_int8"),
        # a prompt of odd length through the whole block at the default expert
        # width of D 1024, fp32 residual stream under bf16 compute
        _case("block", "bf16", 1999, 1024, 16, 2, ffn_dim(1024, 2.67), name="block_prompt_bf16"),
        # a batch of prompts on the int8 weights of the decode layer
        _case("forward", "int8", 4096, 2048, 64, 8, 1408, name="prefill_int8"),
        # benchmark configuration C2: an ordinary batch on a small layer
        _case("forward", "bf16", 16384, 512, 8, 2, 2048, name="forward_c2"),
        # benchmark configuration C3: skewed routing (Zipf 1.2)
        _case("forward", "bf16", 65536, 1024, 16, 2, 4096, zipf=1.2, name="forward_c3_zipf"),
        # benchmark configuration C4, the headline: many small experts, large batch
        _case("forward", "bf16", 65536, 2048, 64, 8, 1024, name="forward_c4"),
        # training in fp32 (the reference's default compute type), D 512 at its
        # default expert width
        _case("train", "fp32", 4096, 512, 8, 2, ffn_dim(512, 2.67), name="train_fp32"),
        # training at the example width D 544 (no multiple of a tile), geglu
        _case("train", "bf16", 4096, 544, 8, 2, ffn_dim(544, 2.67), etype=GEGLU,
              name="train_d544_geglu"),
        # a training step at C2's sizes and at C4's
        _case("train", "bf16", 16384, 512, 8, 2, 2048, name="train_c2"),
        _case("train", "bf16", 65536, 2048, 64, 8, 1024, name="train_c4"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the ranges the listed ones stand for: decode (1-512
    tokens), prompts and batches (513-32768), whole blocks and training steps;
    widths from 64 to 2048, multiples of a tile and not; every expert kind."""
    while True:
        use = rng.choice(("decode", "batch", "batch", "block", "train", "train"))
        E = rng.choice((4, 8, 8, 16, 32, 64, 128, rng.randint(3, 96)))
        K = min(E, rng.choice((1, 2, 2, 4, 8)))
        D = _log_int(rng, 64, 2048)
        D = {0: D, 1: max(64, D // 32 * 32), 2: max(64, D // 64 * 64),
             3: max(128, D // 128 * 128)}[rng.choice((0, 1, 2, 3, 3))]
        F = rng.choice((ffn_dim(D, 2.67), ffn_dim(D, 2.0), max(64, _log_int(rng, 128, 4096) // 64 * 64)))
        etype = rng.choice((SWIGLU, SWIGLU, SWIGLU, GEGLU, MLP))
        act = rng.choice((SILU, GELU, RELU, LEAKY_RELU_SQ)) if etype == MLP else (GELU if etype == GEGLU else SILU)
        zipf = rng.choice((0.0, 0.0, 0.0, round(rng.uniform(0.3, 1.3), 2)))
        if use == "decode":
            dtype = rng.choice(("int8", "bf16"))
            c = _case("forward", dtype, _log_int(rng, 1, 512), D, E, K, F, etype, act, zipf)
        elif use == "train":
            dtype = rng.choice(("bf16", "bf16", "fp32"))
            c = _case("train", dtype, _log_int(rng, 512, 32768), D, E, K, F, etype, act, zipf)
        else:
            dtype = rng.choice(("bf16", "bf16", "int8", "fp32"))
            c = _case("block" if use == "block" else "forward", dtype, _log_int(rng, 513, 32768),
                      D, E, K, F, etype, act, zipf)
        fl, weights = work(c)["flops"], E * 3 * D * F
        if weights > 600e6 or fl > (3e11 if dtype == "fp32" else 4e12):
            continue
        return c


def _wpe(c):
    return 2 if c["etype"] == MLP else 3


def work(c):
    N, D, E, K, F, wpe = c["N"], c["D"], c["E"], c["K"], c["F"], _wpe(c)
    train = c["call"] == "train"
    expert = 2.0 * wpe * N * K * D * F
    router = 2.0 * N * D * E
    flops = (expert + router) * (3 if train else 1)
    xb = 2 if c["dtype"] != "fp32" and c["call"] != "block" else 4
    wb = {"fp32": 4, "bf16": 2, "int8": 1}[c["dtype"]]
    used = E * (1.0 - (1.0 - K / E) ** N)  # experts that have a row, at even routing
    rb = 4 if c["dtype"] == "fp32" else 2
    nbytes = N * D * xb + used * wpe * D * F * wb + D * E * rb + N * D * 4
    if c["dtype"] == "int8":
        nbytes += used * (2 * F + D) * 4
    if c["call"] == "block":
        nbytes += 2 * D * 4
    if train:  # the upstream gradient in, dx and the weight gradients out
        nbytes += N * D * 8 + D * E * 4 + E * wpe * D * F * 4
    return {"bytes": float(nbytes), "flops": flops}


def tolerance(c):
    # Four times what the worst output was seen to differ from the 64-bit
    # values: 3.8e-3 under bf16 compute (the roundings of the projections, the
    # hidden and the expert outputs), 1.5e-6 in fp32, 8e-6 for its gradients, whose
    # products carry about 16 bits.  "max" is what the tail of 1e8 such
    # errors reaches, again times four.
    if c["dtype"] == "fp32":
        return {"rel": 3.2e-5, "max": 5e-3} if c["call"] == "train" else {"rel": 6e-6, "max": 3e-4}
    return {"rel": 1.6e-2, "max": 0.2}


def _inputs(c, seed):
    """The inputs of one case, on the GPU: x ~ N(0, 1), weights ~ N(0, 0.02)
    ("weight_init": "normal"), rounded to bf16 where the case computes in it."""
    N, D, E, F, wpe = c["N"], c["D"], c["E"], c["F"], _wpe(c)
    g = torch.Generator(device="cuda").manual_seed(int(seed))

    def randn(*shape):
        return torch.randn(*shape, generator=g, device="cuda", dtype=torch.float32)

    low = c["dtype"] != "fp32"
    x = randn(N, D)
    wr = randn(D, E) * 0.02
    if c["zipf"] > 0:
        # the router has no bias: a constant last feature carries one, the
        # logarithm of the expert's share
        x[:, D - 1] = 1.0
        wr[D - 1] = -c["zipf"] * torch.log(torch.arange(1, E + 1, device="cuda").float())
    out = {}
    if low:
        wr = wr.bfloat16()
        if c["call"] != "block":
            x = x.bfloat16()
    if c["call"] == "block":
        out["norm"] = 1.0 + 0.1 * randn(D)
        out["scale"] = 0.5 + 0.1 * randn(D)
    if c["call"] == "train":
        out["d_delta"] = randn(N, D)
    out["x"], out["wr"] = x, wr
    # [E, in, out] per matrix: (gate, up, down) or (up, down)
    mats = []
    for j in range(wpe):
        rows, cols = (F, D) if j == wpe - 1 else (D, F)
        w = randn(E, rows, cols).mul_(0.02)
        if c["dtype"] == "int8":
            s = w.abs().amax(dim=1) / 127.0
            q = torch.empty(E, rows, cols, dtype=torch.int8, device="cuda")
            for e in range(E):
                q[e] = torch.round(w[e] / s[e]).clamp_(-127, 127).to(torch.int8)
            mats.append((q, s))
        else:
            mats.append(w.bfloat16() if low else w)
        del w
    out["mats"] = mats
    return out


def _ptr(t):
    return types.SimpleNamespace(value=t.data_ptr())


def prepare(c, seed):
    N, D, E, K, F, wpe = c["N"], c["D"], c["E"], c["K"], c["F"], _wpe(c)
    v = _inputs(c, seed)
    torch.cuda.synchronize()  # the op reads the weights on a stream of its own
    flags = (INT8_WEIGHTS if c["dtype"] == "int8" else 0) | (KEEP_FOR_BACKWARD if c["call"] == "train" else 0)
    op = MoEFeedForward([1, N, D, E, K, c["etype"], F, c["act"]], [0.5],
                        compute_dtype="fp32" if c["dtype"] == "fp32" else "bf16", flags=flags)
    lib = mixlab_amd.load()
    wcode = F32 if c["dtype"] == "fp32" else BF16
    op.set_input(1, (_ptr(v["wr"]), wcode, (D, E)))
    for e in range(E):
        for j, m in enumerate(v["mats"]):
            i = 2 + e * wpe + j
            shape = (F, D) if j == wpe - 1 else (D, F)
            if c["dtype"] == "int8":
                q, s = m
                shp = (ctypes.c_int64 * 2)(*shape)
                rc = lib.mxm_moe_set_input_q8(op.handle, i, q[e].data_ptr(), s[e].data_ptr(), shp, 2, 1)
                if rc != 0:
                    raise RuntimeError("mxm_moe_set_input_q8: %d" % rc)
            else:
                op.set_input(i, (_ptr(m[e]), wcode, shape))
    st = {"c": c, "op": op, "lib": lib, "x": v["x"],
          "x_code": BF16 if v["x"].dtype == torch.bfloat16 else F32,
          "out": torch.empty(N, D, device="cuda"), "aux": torch.empty(1, device="cuda"),
          "ent": torch.empty(1, device="cuda")}
    for k in ("norm", "scale", "d_delta"):
        if k in v:
            st[k] = v[k]
    if c["call"] == "train":
        st["dx"] = torch.empty(N, D, device="cuda")
        st["dwr"] = torch.empty(D, E, device="cuda")
        st["dw"] = torch.empty(E, wpe, D * F, device="cuda")
    return st


def run(st):
    op, N = st["op"], st["c"]["N"]
    x, out, aux, ent = (st[k].data_ptr() for k in ("x", "out", "aux", "ent"))
    if st["c"]["call"] == "block":
        op.block_forward(x, st["x_code"], N, st["norm"].data_ptr(), st["scale"].data_ptr(), F32,
                         EPS, AUX_WEIGHT, out, aux, ent)
    else:
        op.forward(x, st["x_code"], N, out, aux, ent)
    res = {"out": st["out"], "aux": st["aux"], "entropy": st["ent"]}
    if st["c"]["call"] == "train":
        rc = st["lib"].mxm_moe_backward_kept(op.handle, st["d_delta"].data_ptr(), D_AUX, D_ENTROPY,
                                             st["dx"].data_ptr(), st["dwr"].data_ptr(),
                                             st["dw"].data_ptr())
        if rc != 0:
            raise RuntimeError("mxm_moe_backward_kept: %d" % rc)
        res.update(dx=st["dx"], d_router=st["dwr"], d_experts=st["dw"])
    return res


def _act(c, g, u):
    if c["etype"] == SWIGLU:
        return torch.sigmoid(g) * u
    if c["etype"] == GEGLU:
        return torch.nn.functional.gelu(g, approximate="tanh") * u
    if c["act"] == SILU:
        return u * torch.sigmoid(u)
    if c["act"] == GELU:
        return torch.nn.functional.gelu(u, approximate="tanh")
    if c["act"] == RELU:
        return torch.relu(u)
    return torch.where(u > 0, u, 0.5 * u) ** 2


def exact(c, seed):
    N, D, E, K, F, wpe = c["N"], c["D"], c["E"], c["K"], c["F"], _wpe(c)
    v = _inputs(c, seed)
    train = c["call"] == "train"
    x0 = v["x"].double()
    x = x0
    if c["call"] == "block":
        x = x0 * torch.rsqrt((x0 * x0).mean(dim=1, keepdim=True) + EPS)
        if c["dtype"] != "fp32":  # scales and normalised rows are bf16 values under bf16 compute
            x = (x * v["norm"].double()).bfloat16().double()
        else:
            x = x * v["norm"].double()
    wr = v["wr"].double()
    if train:
        x.requires_grad_(True)
        wr.requires_grad_(True)
    # under bf16 compute the logits and the probabilities are bf16 values, as
    # every product of two bf16 tensors is: it is among those that the K
    # largest are picked, equal ones by the lower expert
    def flow(t):
        return t + (t.detach().bfloat16().double() - t.detach()) if c["dtype"] != "fp32" else t

    p = flow(torch.softmax(flow(x @ wr), dim=1))
    idx = torch.sort(p.detach(), dim=1, descending=True, stable=True).indices[:, :K]
    tp = p.gather(1, idx)
    gates = tp / tp.sum(dim=1, keepdim=True).clamp_min(1e-12)
    load = torch.bincount(idx.reshape(-1), minlength=E).double() / (K * N)
    aux = E * (p.mean(dim=0) * load).sum()
    ent = -(p * torch.log(p.clamp_min(1e-12))).sum(dim=1).mean()

    def matrix(e, j):
        m = v["mats"][j]
        return m[0][e].double() * m[1][e].double() if c["dtype"] == "int8" else m[e].double()

    delta = torch.zeros(N, D, dtype=torch.float64, device="cuda")
    xd, gd = x.detach(), gates.detach()
    dx = torch.zeros_like(delta) if train else None
    dgate = torch.zeros(N, K, dtype=torch.float64, device="cuda") if train else None
    dw = torch.zeros(E, wpe, D * F, dtype=torch.float64, device="cuda") if train else None
    for e in range(E):
        rows, place = (idx == e).nonzero(as_tuple=True)
        if not rows.numel():
            continue
        ws = [matrix(e, j) for j in range(wpe)]
        xe = xd[rows]
        if train:
            xe.requires_grad_(True)
            for w in ws:
                w.requires_grad_(True)
        u = xe @ ws[-2]
        g = xe @ ws[0] if wpe == 3 else None
        y = _act(c, g, u) @ ws[-1]
        gate = gd[rows, place].unsqueeze(1)
        delta.index_add_(0, rows, y.detach() * gate)
        if train:
            dd = v["d_delta"][rows].double()
            dgate[rows, place] = (dd * y.detach()).sum(dim=1)
            y.backward(dd * gate)
            dx.index_add_(0, rows, xe.grad)
            for j, w in enumerate(ws):
                dw[e, j] = w.grad.reshape(-1)
    res = {"out": delta, "aux": aux.detach().reshape(1), "entropy": ent.detach().reshape(1)}
    if c["call"] == "block":
        res["out"] = x0 + delta * v["scale"].double()
        res["aux"] = res["aux"] * AUX_WEIGHT
    if train:
        ((gates * dgate).sum() + D_AUX * aux + D_ENTROPY * ent).backward()
        res.update(dx=dx + x.grad, d_router=wr.grad, d_experts=dw)
    return res
