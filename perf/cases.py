"""The calls this library is timed on, through its public entry points.

Six operators carry the path: the Mamba-1 selective scan, the Mamba-2 SSD chunk scan, the Mamba-2
decode step, the four-path 2D scan, the causal conv1d ahead of a scan and the gated RMSNorm after
it.  The listed cases are the layers those run in: training steps (forward and every gradient) and
prompts or tokens at inference (forward alone), from a single token of one sequence to a whole
2.8B-layer batch.  ``draw`` gives further sizes of the same ranges, ragged ones included.

A case is a dict: ``op``, its sizes, the activations' ``dtype`` ("bf16", "f16" or "f32") and
``train`` (forward and backward, against forward alone without autograd).  Inputs follow the
distributions of the operators' benchmark: activations N(0, 1), step sizes
softplus(N(0, 1) + log(expm1(U(1e-3, 1e-1)))) in float32, S4D-real A for Mamba-1 and -U(1, 16) per
head for Mamba-2, float32 parameters.
"""

import math
import os
import sys

import torch
import torch.nn.functional as F

sys.path.insert(0, os.path.join(os.getcwd(), "metal-kernelops_amd"))

DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}


def listed():
    return [
        # Training one Mamba-1 layer of the 2.8B and of the 130M model: the largest calls, and the
        # benchmark's own.
        mamba1("mamba1_train_2.8b", 4, 5120, 4096, "bf16", True),
        mamba1("mamba1_train_130m", 8, 1536, 2048, "bf16", True),
        # One user's prompt through a 2.8B layer: one sequence, of no round length, no gradients.
        mamba1("mamba1_prompt", 1, 5120, 1003, "bf16", False),
        # Training one Mamba-2 layer: the benchmark's head shape.
        ssd("ssd_train", 4, 4096, 64, 64, 1, 128, "bf16", True, False),
        # Float32 training with grouped B and C (32 heads in 8 groups).
        ssd("ssd_train_f32", 4, 1024, 32, 64, 8, 128, "f32", True, False),
        # One user's next turn through a 130M layer: 24 heads, a ragged length, the state carried in.
        ssd("ssd_prompt", 1, 1999, 24, 64, 1, 128, "bf16", False, True),
        # One token of one sequence through a 1.3B layer: the smallest call, all latency.
        decode("decode_one", 1, 16, 128, 128, 1, "f32"),
        # One token of a full serving batch through a 2.7B layer.
        decode("decode_batch", 256, 80, 64, 128, 1, "bf16"),
        # Training a VMamba stage on one image: many short rows, four paths.
        ss2d("ss2d_train", 1, 96, 1, 16, 56, 56, "f32", True),
        # The convolution ahead of the 2.8B layer's scan.
        conv("conv_train", 4, 5120, 4096, 4, "bf16", True),
        # The norm after a 2.7B Mamba-2 layer's scan, gate before the norm as that block has it.
        norm("norm_train", 8192, 5120, 5120, "bf16", True, False),
    ]


def mamba1(name, batch, dim, length, dtype, train, dstate=16, groups=1):
    return {"name": name, "op": "mamba1", "batch": batch, "dim": dim, "length": length, "dstate": dstate,
            "groups": groups, "dtype": dtype, "train": train}


def ssd(name, batch, length, heads, headdim, groups, dstate, dtype, train, carried):
    return {"name": name, "op": "ssd", "batch": batch, "length": length, "heads": heads, "headdim": headdim,
            "groups": groups, "dstate": dstate, "dtype": dtype, "train": train, "carried": carried}


def decode(name, batch, heads, headdim, dstate, groups, dtype):
    return {"name": name, "op": "decode", "batch": batch, "heads": heads, "headdim": headdim, "dstate": dstate,
            "groups": groups, "dtype": dtype, "train": False}


def ss2d(name, batch, channels, groups, dstate, height, width, dtype, train):
    return {"name": name, "op": "ss2d", "batch": batch, "channels": channels, "groups": groups, "dstate": dstate,
            "height": height, "width": width, "dtype": dtype, "train": train}


def conv(name, batch, channels, length, taps, dtype, train):
    return {"name": name, "op": "conv", "batch": batch, "channels": channels, "length": length, "taps": taps,
            "dtype": dtype, "train": train}


def norm(name, rows, features, group, dtype, train, norm_first):
    return {"name": name, "op": "norm", "rows": rows, "features": features, "group": group, "dtype": dtype,
            "train": train, "norm_first": norm_first}


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """A further case: the operators by how much of the path they are, the sizes of real layers with
    batch and length spread over their logarithms, mostly 16-bit activations."""
    op = rng.choice(["mamba1"] * 4 + ["ssd"] * 5 + ["decode"] * 2 + ["ss2d", "conv", "norm"])
    dtype = rng.choice(["bf16", "bf16", "bf16", "f16", "f32"])
    train = rng.random() < 0.6
    while True:
        if op == "mamba1":
            dim = rng.choice([768, 1536, 2048, 3072, 4096, 5120])
            case = mamba1("", rng.choice([1, 1, 2, 3, 4, 8]), dim, _log_int(rng, 64, 4096), dtype, train,
                          rng.choice([16, 16, 16, 8]), rng.choice([1, 1, 1, 2]))
            if rng.random() < 0.5:
                case["length"] = max(64, case["length"] // 64 * 64)
            size, most = case["batch"] * dim * case["length"], 4 * 5120 * 4096
        elif op == "ssd":
            heads, groups = rng.choice([(24, 1), (32, 1), (32, 8), (48, 1), (64, 1), (80, 1), (16, 2)])
            case = ssd("", rng.choice([1, 1, 2, 3, 4, 8]), _log_int(rng, 64, 4096), heads,
                       rng.choice([64, 64, 64, 128]), groups, rng.choice([128, 128, 64]), dtype, train,
                       rng.random() < 0.3)
            if rng.random() < 0.5:
                case["length"] = max(64, case["length"] // 64 * 64)
            size = case["batch"] * case["length"] * heads * case["headdim"] * (4 if dtype == "f32" else 1)
            most = 4 * 4096 * 64 * 64
        elif op == "decode":
            heads = rng.choice([16, 24, 32, 64, 80])
            case = decode("", _log_int(rng, 1, 256), heads, rng.choice([64, 64, 128]), rng.choice([128, 128, 64]), 1,
                          dtype)
            size, most = case["batch"] * heads * case["headdim"] * case["dstate"], 256 * 80 * 64 * 128
        elif op == "ss2d":
            side = rng.choice([14, 28, 56])
            case = ss2d("", rng.choice([1, 2, 4]), rng.choice([96, 192, 384]), 1, rng.choice([16, 16, 8]), side,
                        side + rng.choice([0, 0, 1, 4]), dtype, train)
            size, most = case["batch"] * case["channels"] * side * case["width"], 4 * 96 * 56 * 56
        elif op == "conv":
            channels = rng.choice([1536, 1792, 3072, 5120, 5376])
            case = conv("", rng.choice([1, 2, 4, 8]), channels, _log_int(rng, 64, 4096), 4, dtype, train)
            size = case["batch"] * channels * case["length"] * (2 if dtype == "f32" else 1)
            most = 4 * 5120 * 4096
        else:
            features = rng.choice([1536, 2560, 4096, 5120])
            case = norm("", _log_int(rng, 1, 8192), features, features // rng.choice([1, 1, 8]), dtype, train,
                        rng.random() < 0.5)
            size, most = case["rows"] * features * (2 if dtype == "f32" else 1), 8192 * 5120
        if size <= most:
            del case["name"]
            return case


# ------------------------------------------------------------------------------------- inputs


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    act = DTYPES[case["dtype"]]

    def randn(*shape, dtype=act):
        return torch.randn(shape, generator=gen, device="cuda").to(dtype)

    def uniform(shape, lo, hi):
        return lo + (hi - lo) * torch.rand(shape, generator=gen, device="cuda")

    def step_bias(n):
        return torch.log(torch.expm1(uniform((n,), 1e-3, 1e-1)))

    op, f32 = case["op"], torch.float32
    if op == "mamba1":
        b, d, length, n, g = (case[k] for k in ("batch", "dim", "length", "dstate", "groups"))
        A = -torch.arange(1, n + 1, dtype=f32, device="cuda").expand(d, n).contiguous()
        args = {"u": randn(b, d, length), "dt": randn(b, d, length, dtype=f32), "A": A, "B": randn(b, g, n, length),
                "C": randn(b, g, n, length), "D": 1.0 + 0.1 * randn(d, dtype=f32), "z": randn(b, d, length),
                "delta_bias": step_bias(d)}
        grads = [randn(b, d, length)]
    elif op == "ssd":
        b, length, h, p, g, n = (case[k] for k in ("batch", "length", "heads", "headdim", "groups", "dstate"))
        args = {"x": randn(b, length, h, p), "dt": randn(b, length, h, dtype=f32), "A": -uniform((h,), 1.0, 16.0),
                "B": randn(b, length, g, n), "C": randn(b, length, g, n), "D": torch.ones(h, device="cuda"),
                "z": randn(b, length, h, p), "dt_bias": step_bias(h)}
        if case["carried"]:
            args["initial_states"] = (0.1 * randn(b, h, p, n, dtype=f32)).to(act)
        grads = [randn(b, length, h, p), (0.1 * randn(b, h, p, n, dtype=f32)).to(act)]
    elif op == "decode":
        b, h, p, n, g = (case[k] for k in ("batch", "heads", "headdim", "dstate", "groups"))
        state = 0.1 * randn(b, h, p, n, dtype=f32)
        # the next state goes into the buffer a decode loop alternates with
        args = {"state": state, "x": randn(b, h, p), "dt": randn(b, h, dtype=f32), "A": -uniform((h,), 1.0, 16.0),
                "B": randn(b, g, n), "C": randn(b, g, n), "D": torch.ones(h, device="cuda"), "z": randn(b, h, p),
                "dt_bias": step_bias(h)}
        return {"case": case, "args": args, "next": torch.empty_like(state)}
    elif op == "ss2d":
        b, c, g, n, height, width = (case[k] for k in ("batch", "channels", "groups", "dstate", "height", "width"))
        A = -torch.arange(1, n + 1, dtype=f32, device="cuda").expand(c, n).contiguous()
        args = {"u": randn(b, c, height, width),
                "dt": F.softplus(randn(b, c, height, width, dtype=f32) + step_bias(c)[:, None, None]), "A": A,
                "B": randn(b, g, n, height, width), "C": randn(b, g, n, height, width)}
        grads = [randn(b, c, height, width)]
    elif op == "conv":
        b, c, length, k = (case[k] for k in ("batch", "channels", "length", "taps"))
        bound = 1.0 / math.sqrt(k)  # nn.Conv1d's own initialisation
        args = {"x": randn(b, c, length), "weight": uniform((c, k), -bound, bound).to(act),
                "bias": uniform((c,), -bound, bound).to(act)}
        grads = [randn(b, c, length)]
    else:
        rows, features = case["rows"], case["features"]
        args = {"x": randn(rows, features), "weight": 1.0 + 0.1 * randn(features, dtype=f32), "z": randn(rows, features)}
        grads = [randn(rows, features)]
    if case["train"]:
        for t in args.values():
            t.requires_grad_(True)
    return {"case": case, "args": args, "grads": grads}


# ------------------------------------------------------------------------------------- the calls


def _forward(state):
    import metal_kernelops as mko
    from metal_kernelops import cv
    case, args = state["case"], state["args"]
    op = case["op"]
    if op == "mamba1":
        return (mko.selective_scan(**args, delta_softplus=True),)
    if op == "ssd":
        return cv.mamba2_chunk_scan(**args, chunk_size=256, dt_softplus=True)
    if op == "decode":
        return cv.mamba2_state_update(**args, dt_softplus=True, out_state=state["next"])
    if op == "ss2d":
        return (cv.ss2d_scan(**args),)
    if op == "conv":
        return (cv.causal_conv1d_fn(**args, activation="silu"),)
    return (cv.rmsnorm_gated(**args, group_size=case["group"], norm_before_gate=case["norm_first"]),)


def run(state):
    if not state["case"]["train"]:
        with torch.no_grad():
            return list(_forward(state))
    outs = list(_forward(state))
    return outs + list(torch.autograd.grad(outs, list(state["args"].values()), state["grads"]))


# ------------------------------------------------------------------------------------- its work


def _item(case):
    return 4 if case["dtype"] == "f32" else 2


def work(case):
    """Every input read once and every output written once in each direction, and the operations of
    the recurrence (for the SSD, of its 64-token block form, causal half only)."""
    s, op, train = _item(case), case["op"], case["train"]
    if op == "mamba1":
        e = case["batch"] * case["dim"] * case["length"]
        bc = 2 * case["batch"] * case["groups"] * case["dstate"] * case["length"] * s
        # per element and state: the decay's product and exponential, the input's product, two
        # multiply-adds; the backward recomputes the first four and adds nine of its own
        flops = e * case["dstate"] * (7 + (20 if train else 0))
        return {"bytes": e * (3 * s + 4) + bc + (e * (5 * s + 8) + 2 * bc if train else 0), "flops": flops}
    if op == "ssd":
        tokens = case["batch"] * case["length"]
        h, p, g, n = case["heads"], case["headdim"], case["groups"], case["dstate"]
        rows, bc = tokens * h * p * s, 2 * tokens * g * n * s
        state = case["batch"] * h * p * n * s
        forward = 3 * rows + bc + tokens * h * 4 + state * (2 if case["carried"] else 1)
        flops = tokens * (h * (p * 65 + 4 * n * p) + g * n * 65)
        if not train:
            return {"bytes": forward, "flops": flops}
        backward = 5 * rows + 2 * bc + tokens * h * 8 + state * (3 if case["carried"] else 1)
        return {"bytes": forward + backward, "flops": 3 * flops}
    if op == "decode":
        h, p, n = case["heads"], case["headdim"], case["dstate"]
        state = case["batch"] * h * p * n
        token = case["batch"] * (3 * h * p * s + 2 * case["groups"] * n * s + 4 * h)
        return {"bytes": 8 * state + token, "flops": 5 * state}
    if op == "ss2d":
        e = case["batch"] * case["channels"] * case["height"] * case["width"]
        bc = 2 * case["batch"] * case["groups"] * case["dstate"] * case["height"] * case["width"] * s
        flops = 4 * e * case["dstate"] * (7 + (20 if train else 0))
        return {"bytes": e * (2 * s + 4) + bc + (e * (3 * s + 8) + 2 * bc if train else 0), "flops": flops}
    if op == "conv":
        e, k = case["batch"] * case["channels"] * case["length"], case["taps"]
        return {"bytes": e * s * (5 if train else 2), "flops": e * (2 * k + 4) * (4 if train else 1)}
    e = case["rows"] * case["features"]
    return {"bytes": e * s * (8 if train else 3), "flops": e * (30 if train else 10)}


def tolerance(case):
    # About four times the largest relative error against 64 bits over the listed and some forty drawn
    # cases: 16-bit results sit at the rounding of what is stored, the SSD's also at its 16-bit
    # operands' (its dA most), and a decode step is float32 throughout.
    if case["op"] == "ssd":
        return {"rel": {"f32": 4e-5, "f16": 4e-3, "bf16": 3e-2}[case["dtype"]]}
    if case["dtype"] == "f32" or case["op"] == "decode":
        return {"rel": 1e-5}
    return {"rel": 1e-2 if case["dtype"] == "bf16" else 2e-3}


# ------------------------------------------------------------------------------------- in 64 bits


def exact(case, seed):
    state = prepare(case, seed)
    args = {k: v.detach().double() for k, v in state["args"].items()}
    op = case["op"]
    if op == "mamba1":
        dt = args["dt"] + args["delta_bias"][:, None]
        got = _scan64(args["u"], F.softplus(dt), args["A"], args["B"], args["C"], args["D"], args["z"],
                      state["grads"][0].double() if case["train"] else None)
        if case["train"]:
            ddt = got[2] * torch.sigmoid(dt)  # softplus's slope
            got = got[:2] + [ddt] + got[3:] + [ddt.sum((0, 2))]
        return got
    if op == "ss2d":
        return _ss2d64(args, state["grads"][0].double() if case["train"] else None)
    if case["train"]:
        for t in args.values():
            t.requires_grad_(True)
    with torch.set_grad_enabled(case["train"]):
        if op == "ssd":
            outs = _ssd64(**args)
        elif op == "decode":
            outs = _decode64(**args)
        elif op == "conv":
            length, k = case["length"], case["taps"]
            padded = F.pad(args["x"], (k - 1, 0))
            pre = sum(padded[..., j:j + length] * args["weight"][:, j, None] for j in range(k))
            outs = [F.silu(pre + args["bias"][:, None])]
        else:
            gate = F.silu(args["z"])
            x = args["x"] if case["norm_first"] else args["x"] * gate
            g = x.reshape(case["rows"], -1, case["group"])
            y = (g * torch.rsqrt(g.square().mean(-1, keepdim=True) + 1e-5)).reshape(x.shape) * args["weight"]
            outs = [y * gate if case["norm_first"] else y]
    if not case["train"]:
        return list(outs)
    grads = torch.autograd.grad(outs, list(args.values()), [g.double() for g in state["grads"]])
    return [t.detach() for t in outs] + list(grads)


def _scan64(u, dt, A, B, C, D, z, dout):
    """The Mamba-1 recurrence step by step and, with ``dout``, its analytic backward: the output, then
    the gradients of u, dt, A, B, C, D and z (those of D and z only when they are given)."""
    b, d, length = u.shape
    g, n = B.shape[1:3]
    per = d // g

    def steps(t):  # time first, channels by group
        return t.permute(2, 0, 1).reshape(length, b, g, per, 1).contiguous()

    us, dts = steps(u), steps(dt)
    Bs, Cs = (t.permute(3, 0, 1, 2).unsqueeze(3).contiguous() for t in (B, C))
    Ag = A.view(g, per, n)
    h = u.new_zeros(b, g, per, n)
    y, hs = torch.empty_like(us), []
    for t in range(length):
        if dout is not None:
            hs.append(h)
        h = torch.exp(dts[t] * Ag) * h + dts[t] * us[t] * Bs[t]
        y[t] = (h * Cs[t]).sum(-1, keepdim=True)
    y = y.view(length, b, d).permute(1, 2, 0)
    if D is not None:
        y = y + u * D[:, None]
    if z is not None:
        sig = torch.sigmoid(z)
    out = y if z is None else y * z * sig
    if dout is None:
        return [out]
    gy = dout if z is None else dout * z * sig
    gs = steps(gy)
    ddu, ddt, dB, dC = torch.empty_like(us), torch.empty_like(us), torch.empty_like(Bs), torch.empty_like(Cs)
    dA, carry = torch.zeros_like(Ag), torch.zeros_like(h)
    for t in reversed(range(length)):
        before = hs.pop()
        bar = gs[t] * Cs[t] + carry
        dC[t] = (gs[t] * h).sum(2, keepdim=True)
        dB[t] = (bar * dts[t] * us[t]).sum(2, keepdim=True)
        ddu[t] = (bar * Bs[t]).sum(-1, keepdim=True)
        carry = torch.exp(dts[t] * Ag) * bar
        through = carry * before
        ddt[t] = (through * Ag).sum(-1, keepdim=True)
        dA += (through * dts[t]).sum(0)
        h = before
    ddu, ddt = (t.view(length, b, d).permute(1, 2, 0) for t in (ddu, ddt))
    dB, dC = (t.squeeze(3).permute(1, 2, 3, 0) for t in (dB, dC))
    du = ddu * dt
    grads = [du if D is None else du + gy * D[:, None], ddt + ddu * u, dA.view(d, n), dB, dC]
    if D is not None:
        grads.append((gy * u).sum((0, 2)))
    if z is not None:
        grads.append(dout * y * sig * (1 + z * (1 - sig)))
    return [out] + grads


def _ss2d64(args, dout):
    u, B = args["u"], args["B"]
    b, c, height, width = u.shape
    g, n = B.shape[1:3]
    length = height * width
    down = torch.arange(length, device=u.device).view(height, width).t().reshape(-1)
    rows = torch.arange(length, device=u.device)
    orders = [rows, down, rows.flip(0), down.flip(0)]

    def stacked(t, lead):
        flat = t.reshape(b, lead, length)
        return torch.cat([flat[..., order] for order in orders], 1)

    def folded(t):
        t = t.reshape(b, 4, -1, length)
        back = [t[:, k][..., torch.argsort(order)] for k, order in enumerate(orders)]
        return (back[0] + back[2]) + (back[1] + back[3])

    got = _scan64(stacked(u, c), stacked(args["dt"], c), args["A"].repeat(4, 1),
                  stacked(B, g * n).view(b, 4 * g, n, length), stacked(args["C"], g * n).view(b, 4 * g, n, length),
                  None, None, None if dout is None else stacked(dout, c))
    out = [folded(got[0]).view(u.shape)]
    if dout is None:
        return out
    _, du, ddt, dA, dB, dC = got
    return out + [folded(du).view(u.shape), folded(ddt).view(u.shape), dA.view(4, c, n).sum(0),
                  folded(dB).view(B.shape), folded(dC).view(B.shape)]


def _ssd64(x, dt, A, B, C, D, z, dt_bias, initial_states=None):
    """The SSD in 64-token blocks, the state carried from block to block."""
    b, length, h, p = x.shape
    g, n = B.shape[2:]
    q, heads = 64, h // g
    blocks = -(-length // q)
    pad = blocks * q - length
    step = F.softplus(dt + dt_bias)

    def cut(t, *tail):  # padded tokens have a step of zero: no decay, no input
        t = F.pad(t, (0, 0) * (t.dim() - 2) + (0, pad))
        return t.reshape(b, blocks, q, *tail)

    u, Bb, Cb = cut(x * step[..., None], g, heads, p), cut(B, g, n), cut(C, g, n)
    cs = torch.cumsum(cut(step * A, g, heads), 2).permute(0, 1, 3, 4, 2)           # (b, block, g, head, q)
    lower = torch.ones(q, q, dtype=torch.bool, device=x.device).tril()
    decay = torch.exp((cs[..., :, None] - cs[..., None, :]).masked_fill(~lower, float("-inf")))
    scores = torch.einsum("bclgn,bcsgn->bcgls", Cb, Bb)
    intra = torch.einsum("bcghls,bcsghp->bclghp", decay * scores.unsqueeze(3), u)
    to_end = torch.exp(cs[..., -1:] - cs).permute(0, 1, 4, 2, 3)
    local = torch.einsum("bcsghp,bcsgn->bcghpn", u * to_end.unsqueeze(-1), Bb)
    state = x.new_zeros(b, g, heads, p, n) if initial_states is None else initial_states.view(b, g, heads, p, n)
    entering = []
    for c in range(blocks):
        entering.append(state)
        state = torch.exp(cs[:, c, :, :, -1])[..., None, None] * state + local[:, c]
    entering = torch.stack(entering, 1)
    inter = torch.einsum("bclgn,bcghpn->bclghp", Cb, entering) * torch.exp(cs).permute(0, 1, 4, 2, 3).unsqueeze(-1)
    y = (intra + inter).reshape(b, blocks * q, h, p)[:, :length] + x * D[:, None]
    return [y * F.silu(z), state.reshape(b, h, p, n)]


def _decode64(state, x, dt, A, B, C, D, z, dt_bias):
    heads = state.shape[1] // B.shape[1]
    step = F.softplus(dt + dt_bias)
    Bh, Ch = (t.repeat_interleave(heads, 1).unsqueeze(2) for t in (B, C))
    state = torch.exp(step * A)[..., None, None] * state + (step[..., None] * x).unsqueeze(-1) * Bh
    y = (state * Ch).sum(-1) + x * D[:, None]
    return [y * F.silu(z), state]
