"""The work that users of this package have it do, as measurable cases.

A case is one pass through public entry points at one set of sizes:

  read        the routed fast-weight read of one layer and chunk without
              gradients (prefill): uttt_amd.moe.apply_moe_fast_weights_grouped
  read_train  the same read with its backward: gradients of the tokens and of
              the expert pool
  update      the aggregate UPDATE of a chunk's writer layers (routing of all
              writers, one grouped update) and its backward: gradients of
              k, v, lr, the gates and the pool
  write       the pool's write: momentum, Newton-Schulz and the
              norm-preserving projection (uttt_amd.fast_weight_write)
  decode      generation: router and read of a few tokens per sequence, each
              sequence with its own pool (uttt_amd.decode)
  dense       a chunk of uTTT-Dense: every layer's read, then the aggregate
              write with momentum and Newton-Schulz (uttt_amd.dense)
  permute     permute by expert, unpermute, and both backward passes
  preprocess  the update inputs' silu, norms and rotary embedding with their
              backward (uttt_amd.moe.preprocess_update_inputs)

The sizes are those of the uTTT configurations: the shipped uTTT-MoE 124M (48
experts, top-1, four heads of 192, expert width 192, chunks of 4096), the
shipped 760M's pool (96 experts, top-1, hidden size 1536 in four heads), the
two benchmark pools (16 experts of 768 x 1536 and 32 of 1536 x 3072, top-2,
chunks of 2048), uTTT-Dense 124M (four heads of 192, r = 2, 12 layers) and
the permute benchmark (65 536 tokens of 768 over 16 experts); draw() spreads
the token counts over the range between a short prompt and a full chunk and
takes odd ones too.
"""
from __future__ import annotations

import math

import torch

BF16 = torch.bfloat16
# expert pools: D, I = the expert's input and inner width, E experts, top-k,
# H fast-weight heads per token
POOLS = {
    "shipped124m": dict(D=192, I=192, E=48, k=1, H=4),
    "shipped760m": dict(D=384, I=384, E=96, k=1, H=4),
    "moe124m": dict(D=768, I=1536, E=16, k=2, H=1),
    "moe760m": dict(D=1536, I=3072, E=32, k=2, H=1),
}
ROPE = 64   # features of one rotary block
NS5 = [(4.0848, -6.8946, 2.9270), (3.9505, -6.3029, 2.6377), (3.7418, -5.5913, 2.3037),
       (2.8769, -3.1427, 1.2046), (2.8366, -3.0525, 1.2012)]


def listed():
    return [
        # a layer-chunk's read of the shipped 124M model: 4096 tokens of four heads
        dict(name="read_shipped124m", op="read", pool="shipped124m", B=1, L=4096),
        # a layer-chunk's read of the 760M benchmark pool (skewed routing)
        dict(name="read_moe760m", op="read", pool="moe760m", B=1, L=2048),
        # the rest of a prompt that does not fill a chunk: ragged, two sequences
        dict(name="read_tail_moe124m", op="read", pool="moe124m", B=2, L=517),
        # a training step's read of the shipped 760M pool, forward and backward
        dict(name="read_train_shipped760m", op="read_train", pool="shipped760m", B=1, L=4096),
        # a training step's aggregate update over the 12 layers of the 124M model
        dict(name="update_shipped124m", op="update", pool="shipped124m", W=12, L=4096),
        # the same of one writer's odd-length chunk at the 124M benchmark pool
        dict(name="update_odd_moe124m", op="update", pool="moe124m", W=1, L=1531),
        # a training step's aggregate update at 760M: 24 writers of 2048 tokens
        dict(name="update_moe760m", op="update", pool="moe760m", W=24, L=2048),
        # the shipped write of the shipped 760M pool: 288 matrices of 384 x 384
        dict(name="write_shipped760m", op="write", pool="shipped760m", muon=True),
        # one generated token of eight sequences, one layer
        dict(name="decode_moe760m", op="decode", pool="moe760m", B=8, T=1),
        # a chunk of uTTT-Dense 124M with the shipped write
        dict(name="dense124m_chunk", op="dense", layers=12, B=1, L=2048, H=4, d=192, r=2, muon=True),
        # permute / unpermute and their backward at the permute benchmark's size
        dict(name="permute_64k", op="permute", T=65536, E=16, k=2, D=768),
        # a layer-chunk's k / v preprocessing at 760M, forward and backward
        dict(name="preprocess_760m", op="preprocess", B=1, L=4096, D=1536, H=4),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["read", "read", "read_train", "update", "update", "write", "decode", "dense",
                     "permute", "preprocess"])
    pool = rng.choice(sorted(POOLS))
    full = 4096 if POOLS[pool]["H"] > 1 else 2048
    if op == "read":
        return dict(op=op, pool=pool, B=rng.choice([1, 1, 2]), L=_log(rng, 65, full))
    if op == "read_train":
        return dict(op=op, pool=pool, B=1, L=_log(rng, 200, full))
    if op == "update":
        return dict(op=op, pool=pool, W=rng.choice([1, 2, 6, 12]), L=_log(rng, 200, full))
    if op == "write":
        return dict(op=op, pool=rng.choice(["shipped124m", "shipped760m", "moe124m"]),
                    muon=rng.random() < 0.7)
    if op == "decode":
        return dict(op=op, pool=pool, B=rng.randint(1, 8), T=rng.choice([1, 1, 2, 3, 4]))
    if op == "dense":
        return dict(op=op, layers=rng.choice([1, 6, 12]), B=1, L=_log(rng, 128, 2048), H=4,
                    d=rng.choice([96, 128, 192]), r=rng.choice([1, 2]), muon=rng.random() < 0.7)
    if op == "permute":
        return dict(op=op, T=_log(rng, 1000, 65536), E=rng.choice([16, 32, 48]),
                    k=rng.choice([1, 2]), D=rng.choice([192, 384, 768]))
    return dict(op="preprocess", B=1, L=_log(rng, 200, 4096), D=rng.choice([768, 1536]), H=4)


# ---------------------------------------------------------------- inputs ----
def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _randn(g, *shape, scale=1.0, dtype=BF16):
    return (torch.randn(*shape, generator=g, device="cuda") * scale).to(dtype)


def _unit(g, *shape):
    t = torch.randn(*shape, generator=g, device="cuda")
    return (t / (t.norm(dim=-1, keepdim=True) + 1e-5)).to(BF16)


def _lr(g, *shape):
    return torch.sigmoid(torch.randn(*shape, generator=g, device="cuda")) * 0.1


def _tokens(g, B, L, H, D):
    """[B, L, H*D] with unit rows per head, as the models normalise q and k."""
    return _unit(g, B, L, H, D).view(B, L, H * D)


def _pool(g, p, B=1):
    W02 = _randn(g, B, p["E"], 2 * p["I"], p["D"], scale=p["D"] ** -0.5)
    W1 = _randn(g, B, p["E"], p["D"], p["I"], scale=p["I"] ** -0.5)
    return W02, W1


def _router(g, p):
    """Router weights (logits ~ N(0, 1) on unit tokens) and the balancing's
    selection bias; the 32-expert pool has a Zipf(1.1) expert prior."""
    R = torch.randn(p["E"], p["D"], generator=g, device="cuda")
    if p["E"] == 32:
        bias = -1.1 * torch.log(torch.arange(p["E"], device="cuda", dtype=torch.float32) + 1)
    else:
        bias = torch.randn(p["E"], generator=g, device="cuda") * 0.5
    return R, bias


def _combine(p):
    return "topk_renorm" if p["k"] > 1 else "selected_prob"


def prepare(case, seed):
    g, op = _gen(seed), case["op"]
    s = dict(case=case)
    if op in ("read", "read_train", "update", "decode", "write"):
        p = s["p"] = POOLS[case["pool"]]
    if op in ("read", "read_train"):
        s["x"] = _tokens(g, case["B"], case["L"], p["H"], p["D"])
        s["W02"], s["W1"] = _pool(g, p, case["B"])
        s["R"], s["bias"] = _router(g, p)
        if op == "read_train":
            s["g"] = _randn(g, *s["x"].shape, scale=0.02)
            s["in"] = [s["x"].requires_grad_(), s["W02"].requires_grad_(), s["W1"].requires_grad_()]
    elif op == "update":
        n = case["W"] * case["L"]
        s["k"] = _tokens(g, 1, n, p["H"], p["D"]).view(1, n * p["H"], p["D"])
        s["v"] = _randn(g, 1, n * p["H"], p["D"], scale=p["D"] ** -0.5)
        s["lr"] = _lr(g, 1, n * p["H"], 3)
        s["W02"], s["W1"] = _pool(g, p)
        s["R"], s["bias"] = _router(g, p)
        s["G"] = [_randn(g, *s["W02"].shape, scale=0.02), _randn(g, *s["W1"].shape, scale=0.02)]
        for n in ("k", "v", "lr", "W02", "W1"):
            s[n].requires_grad_()
    elif op == "write":
        s["grads"], s["masters"], s["mom"] = [], [], []
        for shape, fan in (((1, p["E"], 2 * p["I"], p["D"]), p["D"]),
                           ((1, p["E"], p["D"], p["I"]), p["I"])):
            # summed token gradients: a few strong directions over a flat rest
            u = torch.randn(*shape[:3], 8, generator=g, device="cuda")
            v = torch.randn(*shape[:2], 8, shape[3], generator=g, device="cuda")
            s["grads"].append((u @ v * 0.01 + _randn(g, *shape, scale=0.02, dtype=torch.float32)).to(BF16))
            s["masters"].append(_randn(g, *shape, scale=fan ** -0.5, dtype=torch.float32))
            s["mom"].append(_randn(g, *shape, scale=0.02, dtype=torch.float32))
        s["coeff"] = torch.sigmoid(torch.randn(1, 1, 1, 1, generator=g, device="cuda"))
    elif op == "decode":
        s["x"] = _unit(g, case["B"], case["T"] * p["H"], p["D"])
        s["W02"], s["W1"] = _pool(g, p, case["B"])
        s["R"], s["bias"] = _router(g, p)
    elif op == "dense":
        from uttt_amd import dense

        b, H, d, r = case["B"], case["H"], case["d"], case["r"]
        w0 = _randn(g, b, H, r * d, d, scale=d ** -0.5)
        w2 = _randn(g, b, H, r * d, d, scale=d ** -0.5)
        w1 = _randn(g, b, H, d, r * d, scale=(r * d) ** -0.5)
        s["w"] = (w0, w1, w2)
        for n in ("q", "k", "v"):
            s[n] = [_tokens(g, b, case["L"], H, d) for _ in range(case["layers"])]
        s["lr"] = [_lr(g, b, case["L"], 3 * H) for _ in range(case["layers"])]
        s["m"] = [torch.sigmoid(torch.randn(b, 1, 1, 1, generator=g, device="cuda"))
                  for _ in range(case["layers"])]
        s["bank"] = dense.SharedFastWeights(w0, w1, w2, r, use_momentum=True,
                                            use_moun=case["muon"])
    elif op == "permute":
        T, E, D = case["T"], case["E"], case["D"]
        logits = torch.randn(1, E, T, generator=g, device="cuda")
        bias = torch.randn(1, E, 1, generator=g, device="cuda") * 0.5
        idx = torch.topk(logits + bias, case["k"], dim=1).indices
        s["mask"] = torch.zeros_like(logits, dtype=torch.bool).scatter_(1, idx, True)
        sm = torch.softmax(logits, dim=1) * s["mask"]
        s["probs"] = (sm / sm.sum(dim=1, keepdim=True)).requires_grad_()
        s["x"] = _randn(g, 1, T, D).requires_grad_()
        s["g"] = _randn(g, 1, T, D)
    else:
        B, L, D = case["B"], case["L"], case["D"]
        s["k"] = _randn(g, B, L, D).requires_grad_()
        s["v"] = _randn(g, B, L, D).requires_grad_()
        s["lr"] = _lr(g, B, L, 3)
        s["gk"], s["gv"] = _randn(g, B, L, D), _randn(g, B, L, D)
        from uttt_amd import moe

        s["tables"] = moe.Rope.tables(ROPE, 10000.0, L, "cuda")
    return s


# ------------------------------------------------------------------- run ----
def _read(s):
    from uttt_amd import moe

    p = s["p"]
    cfg = moe.RouterConfig(topk=p["k"], combine_mode=_combine(p))
    return moe.apply_moe_fast_weights_grouped(s["x"], None, s["W1"], None, s["R"], cfg, p["H"],
                                              routing_bias=s["bias"], precomputed_w0_w2=s["W02"])


def run(s):
    op = s["case"]["op"]
    if op == "read":
        with torch.no_grad():
            out, (_, group_sizes) = _read(s)
        return out, group_sizes
    if op == "read_train":
        out, _ = _read(s)
        return (out.detach(),) + torch.autograd.grad(out, s["in"], s["g"])
    if op == "update":
        from uttt_amd import moe

        p = s["p"]
        cfg = moe.RouterConfig(topk=p["k"], combine_mode=_combine(p))
        with torch.no_grad():
            mask, _, probs, _ = moe.route_writers(s["k"].detach(), s["case"]["W"], s["R"], cfg,
                                                  routing_bias=s["bias"])
        probs.requires_grad_()
        dW = moe.aggregate_moe_update_grads(
            [moe.WriterInputs(s["k"], s["v"], s["lr"], mask, probs)], None, s["W1"], None, p["k"],
            precomputed_w0_w2=s["W02"], packed=True)
        grads = torch.autograd.grad(dW, [s["k"], s["v"], s["lr"], probs, s["W02"], s["W1"]],
                                    s["G"])
        return (dW[0].detach(), dW[1].detach()) + grads
    if op == "write":
        from uttt_amd import fast_weight_write as fww

        fast, master, mom = fww.apply_moe_update_packed(
            *s["grads"], *s["masters"], momentum_buf=tuple(s["mom"]), m_coeff=s["coeff"],
            use_momentum=True, use_moun=s["case"]["muon"])
        return fast + master + mom
    if op == "decode":
        from uttt_amd import decode

        p = s["p"]
        with torch.no_grad():
            out, _ = decode.apply_moe_fast_weights_decode(
                s["x"], None, s["W1"], None, s["R"], p["k"], routing_bias=s["bias"],
                precomputed_w0_w2=s["W02"], combine_mode=_combine(p))
        return out
    if op == "dense":
        bank = s["bank"]
        out = [bank.read(q) for q in s["q"]]
        bank.write(s["k"], s["v"], s["lr"], momentum_coeffs=s["m"])
        return out + [bank.W02, bank.W1, bank.M02, bank.M1, bank.MOM02, bank.MOM1]
    if op == "permute":
        from uttt_amd.lact_moe_triton import triton_permute as tp

        xp, pp, row_map = tp.permute_with_expert_mask(s["x"], s["mask"], s["probs"], s["case"]["k"])
        y = tp.unpermute_and_merge_with_probs(xp, row_map, s["probs"])
        return (xp.detach(), pp.detach(), y.detach()) + torch.autograd.grad(
            y, [s["x"], s["probs"]], s["g"])
    from uttt_amd import moe

    rope = moe.Rope(*s["tables"])
    k, v, lr = moe.preprocess_update_inputs(s["k"], s["v"], s["lr"], s["case"]["H"],
                                            qkv_silu=True, v_norm=True, qk_norm=True, rope=rope)
    grads = torch.autograd.grad([k, v], [s["k"], s["v"]], [s["gk"].view(k.shape), s["gv"].view(v.shape)])
    return (k.detach(), v.detach(), lr) + grads


# ------------------------------------------------------------------ work ----
def work(case):
    op = case["op"]
    p = POOLS.get(case.get("pool"), {})
    if p:
        D, I, E, k, H = p["D"], p["I"], p["E"], p["k"], p["H"]
        wbytes = 3 * E * D * I * 2
    if op == "read":
        T = case["B"] * case["L"] * H
        return dict(bytes=case["B"] * wbytes + 2 * T * D * 2 + E * D * 4,
                    flops=T * (6 * k * I * D + 2 * E * D))
    if op == "read_train":
        T = case["L"] * H
        # x, g, pool read; out, grad x, grad pool written
        return dict(bytes=2 * wbytes + 4 * T * D * 2 + E * D * 4,
                    flops=T * (18 * k * I * D + 2 * E * D))
    if op == "update":
        T = case["W"] * case["L"] * H
        # pool, upstream gradients, k, v, lr read; dW, pool gradients, grad k, v, lr, gates written
        return dict(bytes=4 * wbytes + 4 * T * D * 2 + 6 * T * 4 + T * E * 4 + E * D * 4,
                    flops=T * (36 * k * I * D + 2 * E * D))
    if op == "write":
        n = 3 * E * D * I
        m, c = min(I, D), max(I, D)
        ns = 3 * E * 5 * (4 * m * m * c + 2 * m ** 3) if case["muon"] else 0
        # gradient, master, momentum read; master, fast weights, momentum written
        return dict(bytes=n * (2 + 4 + 4 + 4 + 2 + 4), flops=ns + 8 * n)
    if op == "decode":
        T = case["T"] * H
        sel = case["B"] * min(E, T * k)
        return dict(bytes=sel * 3 * D * I * 2 + case["B"] * T * D * 4 + E * D * 4,
                    flops=case["B"] * T * (6 * k * I * D + 2 * E * D))
    if op == "dense":
        d, H, r, n = case["d"], case["H"], case["r"], case["layers"] * case["B"] * case["L"]
        w = case["B"] * H * 3 * r * d * d
        ns = case["B"] * H * 3 * r * 5 * 6 * d ** 3 if case["muon"] else 0
        # q, k, v, lr read and the reads written; weights, masters, momentum read and written
        return dict(bytes=n * H * (4 * d * 2 + 12) + w * 20, flops=n * H * 18 * r * d * d + ns)
    if op == "permute":
        T, k, D, E = case["T"], case["k"], case["D"], case["E"]
        # x, mask, probs read, xp written; y written; g read, grad x and grad probs written
        return dict(bytes=T * D * 2 * (4 + k) + T * E * 9 + 4 * k * T, flops=6 * T * k * D)
    n = case["B"] * case["L"] * case["D"]
    return dict(bytes=n * 2 * 8, flops=60 * n)


def tolerance(case):
    op = case["op"]
    if op in ("read", "read_train"):
        # bf16 hidden and expert outputs: 2-4e-3 against 64 bits
        return {"rel": 1.2e-2, "differ": 2e-3}
    if op == "update":
        return {"rel": 2e-2}
    if op == "write":
        # Newton-Schulz keeps bf16 matrices over five iterations; without it
        # only the fast weights' rounding is left
        return {"rel": 2e-2} if case["muon"] else {"rel": 8e-3}
    if op == "dense":
        return {"rel": 2e-2}
    return {"rel": 1.2e-2}


# ----------------------------------------------------------------- exact ----
def _route_exact(s, x, B):
    """Top-k mask and gates [B, T, E] of x [B, T, D] in 64 bits."""
    p = s["p"]
    logits = x @ s["R"].double().T
    idx = torch.topk(logits + s["bias"].double(), p["k"], dim=-1).indices
    mask = torch.zeros_like(logits, dtype=torch.bool).scatter_(-1, idx, True)
    probs = torch.softmax(logits, dim=-1) * mask
    if _combine(p) == "topk_renorm":
        probs = probs / probs.sum(dim=-1, keepdim=True)
    return mask, probs


def _expert(x, W02, W1):
    y0, y2 = (x @ W02.T).chunk(2, dim=-1)
    return (y0 * torch.sigmoid(y0) * y2) @ W1.T


def _read_exact(s, x, W02, W1):
    """The routed read of x [B, T, D] with pools W02 [B][E], W1 [B][E]."""
    mask, probs = _route_exact(s, x.detach(), x.shape[0])
    outs = []
    for b in range(x.shape[0]):
        out = torch.zeros_like(x[b])
        for e in range(s["p"]["E"]):
            t = mask[b, :, e].nonzero(as_tuple=True)[0]
            if t.numel():
                out = out.index_add(0, t, _expert(x[b, t], W02[b][e], W1[b][e]) * probs[b, t, e, None])
        outs.append(out)
    return torch.stack(outs), mask


def _update_expert(k, v, lr, p, W02, W1):
    """dW of one expert's rows: the gradient of the lr-weighted dot products."""
    y0, y2 = (k @ W02.T).chunk(2, dim=-1)
    vp = v * p[:, None]
    dh = vp @ W1
    sg = torch.sigmoid(y0)
    dy0 = lr[:, 0:1] * sg * y2 * dh * (1 + y0 * (1 - sg))
    dy2 = lr[:, 2:3] * sg * y0 * dh
    hid = lr[:, 1:2] * sg * y0 * y2
    return torch.cat([dy0.T @ k, dy2.T @ k]), vp.T @ hid


def _orthogonalise(G, scale=1.0):
    X = G.double()
    wide = X.shape[-2] > X.shape[-1]
    if wide:
        X = X.transpose(-1, -2).contiguous()
    X = X / (X.norm(dim=(-2, -1), keepdim=True) + 1e-7)
    for a, b, c in NS5:
        A = X @ X.transpose(-1, -2).contiguous()
        X = a * X + (b * A + c * (A @ A)) @ X
    return (X.transpose(-1, -2).contiguous() if wide else X) * scale


def _project(master, step, norm):
    new = master + step
    return new / (new.norm(dim=-1, keepdim=True) + 1e-5) * norm


def exact(case, seed):
    s, op = prepare(case, seed), case["op"]
    dbl = torch.Tensor.double
    if op in ("read", "read_train"):
        p, B, L = s["p"], case["B"], case["L"]
        x = dbl(s["x"].detach()).view(B, L * p["H"], p["D"])
        E = p["E"]
        train = op == "read_train"
        if train:
            x.requires_grad_()
        W02 = [[dbl(s["W02"].detach()[b, e]).requires_grad_(train) for e in range(E)] for b in range(B)]
        W1 = [[dbl(s["W1"].detach()[b, e]).requires_grad_(train) for e in range(E)] for b in range(B)]
        out, mask = _read_exact(s, x, W02, W1)
        if not train:
            return out.view(s["x"].shape), None
        flat = [w for ws in W02 + W1 for w in ws]
        gr = torch.autograd.grad(out, [x] + flat, dbl(s["g"]).view(out.shape), allow_unused=True)
        gr = [torch.zeros_like(w) if q is None else q for q, w in zip(gr, [x] + flat)]
        return (out.detach().view(s["x"].shape), gr[0].view(s["x"].shape),
                torch.stack(gr[1:1 + B * E]).view(s["W02"].shape),
                torch.stack(gr[1 + B * E:]).view(s["W1"].shape))
    if op == "update":
        p = s["p"]
        E, D, I = p["E"], p["D"], p["I"]
        k, v, lr = s["k"].detach()[0], s["v"].detach()[0], s["lr"].detach()[0]
        mask, probs = _route_exact(s, dbl(k)[None], 1)
        # the update takes lr in bf16, the fast weights' type
        lr = dbl(lr.to(BF16))
        out = [torch.zeros(1, E, 2 * I, D, dtype=torch.float64, device="cuda"),
               torch.zeros(1, E, D, I, dtype=torch.float64, device="cuda")]
        gk, gv, glr = (torch.zeros(t.shape, dtype=torch.float64, device="cuda") for t in (k, v, lr))
        gp = torch.zeros(1, E, k.shape[0], dtype=torch.float64, device="cuda")
        gw = [torch.zeros_like(o) for o in out]
        for e in range(E):
            t = mask[0, :, e].nonzero(as_tuple=True)[0]
            if not t.numel():
                continue
            ins = [dbl(k[t]), dbl(v[t]), lr[t], probs[0, t, e].detach(),
                   dbl(s["W02"].detach()[0, e]), dbl(s["W1"].detach()[0, e])]
            ins = [i.requires_grad_() for i in ins]
            d = _update_expert(*ins)
            gr = torch.autograd.grad(d, ins, [dbl(s["G"][0][0, e]), dbl(s["G"][1][0, e])])
            out[0][0, e], out[1][0, e] = d[0].detach(), d[1].detach()
            gk.index_add_(0, t, gr[0])
            gv.index_add_(0, t, gr[1])
            glr.index_add_(0, t, gr[2])
            gp[0, e, t] = gr[3]
            gw[0][0, e], gw[1][0, e] = gr[4], gr[5]
        return out[0], out[1], gk[None], gv[None], glr[None], gp, gw[0], gw[1]
    if op == "write":
        p = s["p"]
        fast, mom = [], []
        for i, (g, w, m) in enumerate(zip(s["grads"], s["masters"], s["mom"])):
            g = dbl(g) + dbl(m) * dbl(s["coeff"])
            mom.append(g)
            step = g
            if case["muon"]:
                n = p["E"] * (2 if i == 0 else 1)
                step = _orthogonalise(g.reshape(n, -1, g.shape[-1])).view(g.shape)
            w = dbl(w)
            fast.append(_project(w, step, w.norm(dim=-1, keepdim=True)))
        return tuple(fast) + tuple(fast) + tuple(mom)
    if op == "decode":
        x = dbl(s["x"])
        mask, probs = _route_exact(s, x, case["B"])
        out = torch.zeros_like(x)
        for b, t, e in mask.nonzero().tolist():
            out[b, t] += _expert(x[b, t][None], dbl(s["W02"][b, e]), dbl(s["W1"][b, e]))[0] * probs[b, t, e]
        return out
    if op == "dense":
        b, H, d, r, n = case["B"], case["H"], case["d"], case["r"], case["layers"]
        w0, w1, w2 = (dbl(w) for w in s["w"])
        heads = lambda t: dbl(t).view(b, -1, H, t.shape[-1] // H).transpose(1, 2)
        outs = []
        d0, d1, d2 = torch.zeros_like(w0), torch.zeros_like(w1), torch.zeros_like(w2)
        for l in range(n):
            q = heads(s["q"][l])
            y0 = q @ w0.transpose(-1, -2)
            o = (y0 * torch.sigmoid(y0) * (q @ w2.transpose(-1, -2))) @ w1.transpose(-1, -2)
            outs.append(o.transpose(1, 2).reshape(s["q"][l].shape))
            k, v, lr = heads(s["k"][l]), heads(s["v"][l]), heads(s["lr"][l])
            y0, y2, dh = k @ w0.transpose(-1, -2), k @ w2.transpose(-1, -2), v @ w1
            sg = torch.sigmoid(y0)
            d0 += (lr[..., 0:1] * sg * y2 * dh * (1 + y0 * (1 - sg))).transpose(-1, -2) @ k / n
            d2 += (lr[..., 2:3] * sg * y0 * dh).transpose(-1, -2) @ k / n
            d1 += v.transpose(-1, -2) @ (lr[..., 1:2] * sg * y0 * y2) / n
        new, moms = [], []
        for i, (w, g) in enumerate(((w0, d0), (w1, d1), (w2, d2))):
            # every d x d slice on its own: row blocks of w0 / w2, column blocks of w1
            cut = (lambda t: t.view(b, H, r, d, d)) if i != 1 else (
                lambda t: t.view(b, H, d, r, d).transpose(2, 3))
            step = cut(g)
            if case["muon"]:
                step = _orthogonalise(step)
            m = cut(w) + step
            f = m / (m.norm(dim=-1, keepdim=True) + 1e-5) * cut(w).norm(dim=-1, keepdim=True)
            back = lambda t: (t if i != 1 else t.transpose(2, 3)).reshape(w.shape)
            new.append((back(f), back(m)))
            moms.append(g)
        shape02, shape1 = (b * H, 1, 2 * r * d, d), (b * H, 1, d, r * d)
        pair = lambda a, c: torch.cat([a, c], dim=2).reshape(shape02)
        return outs + [pair(new[0][0], new[2][0]), new[1][0].reshape(shape1),
                       pair(new[0][1], new[2][1]), new[1][1].reshape(shape1),
                       pair(moms[0], moms[2]), moms[1].reshape(shape1)]
    if op == "permute":
        x, g, probs = dbl(s["x"].detach())[0], dbl(s["g"])[0], dbl(s["probs"].detach())[0]
        e, t = s["mask"][0].nonzero(as_tuple=True)          # expert-major, token-ascending
        y = torch.zeros_like(x).index_add_(0, t, x[t] * probs[e, t, None])
        gx = torch.zeros_like(x).index_add_(0, t, g[t] * probs[e, t, None])
        gp = torch.zeros_like(probs)
        gp[e, t] = (g[t] * x[t]).sum(-1)
        return x[t][None], probs[e, t][None], y[None], gx[None], gp[None]
    B, L, D, H = case["B"], case["L"], case["D"], case["H"]
    k, v = dbl(s["k"].detach()).requires_grad_(), dbl(s["v"].detach()).requires_grad_()
    cos, sin = (dbl(t[:L])[None, :, None, :] for t in s["tables"])
    sk = (k * torch.sigmoid(k)).view(B, L, H, D // H)
    sk = sk / (sk.norm(dim=-1, keepdim=True) + 1e-5)
    a, c = sk.view(B, L, D // ROPE, ROPE).chunk(2, dim=-1)
    ko = torch.cat([a * cos - c * sin, c * cos + a * sin], dim=-1).reshape(B, L * H, D // H)
    sv = v * torch.sigmoid(v)
    vo = (sv * torch.rsqrt((sv * sv).mean(-1, keepdim=True) + 1e-5)).reshape(B, L * H, D // H)
    gk, gv = torch.autograd.grad([ko, vo], [k, v], [dbl(s["gk"]).view(ko.shape), dbl(s["gv"]).view(vo.shape)])
    lr = dbl(s["lr"]).repeat_interleave(H, dim=1)
    return ko.detach(), vo.detach(), lr, gk, gv
