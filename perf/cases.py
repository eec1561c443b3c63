"""Performance cases of the scans: what a program that uses this package has it do.

Each case is one pass through the public entry points on tensors already on the GPU:

  fwd, rev            scan_forward on (batch, dim, seqlen) rows, each direction
  train               pscan forward, then its gradients for a given grad_out
  cl_fwd, cl_train    the channel-last forms, (batch, seqlen, dim)
  softplus_fwd, softplus_train
                      the scan whose gates exp(-softplus(z) * rate[d]) are made in the kernels
  dimwise             dimwise_forward on a copy of its input (it works in place)

Inputs are those of a Mamba-style layer: decays exp(-softplus(N(0,1)) * rate) with rates
between 0.001 and 0.1, tokens 0.1 N(0,1), output gradients N(0,1).
"""
import torch

import fpscan_amd

DTYPES = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
SIZE = {"f32": 4, "f16": 2, "bf16": 2}

# groups per chunk and elements per group of dimwise_forward by seqlen
DIMWISE_CHUNK = {64: (2, 32), 128: (4, 32), 256: (8, 32), 512: (16, 32), 1024: (16, 64),
                 2048: (32, 64), 4096: (32, 128), 8192: (32, 128), 16384: (32, 128),
                 32768: (32, 128), 65536: (32, 128)}


def _case(op, dtype, batch, dim, seqlen):
    return {"op": op, "dtype": dtype, "batch": batch, "dim": dim, "seqlen": seqlen}


def listed():
    cases = [
        # a short row scan of the published latency table (fp32, 2 x 256 rows): the call itself
        _case("fwd", "f32", 2, 256, 256),
        # the other direction in half precision, at a long row of the same table
        _case("rev", "f16", 2, 256, 16384),
        # the smallest training step of the benchmark: forward and gradients of 2 MiB tensors
        _case("train", "f32", 2, 256, 1024),
        # a training step of an ordinary layer (32 MiB tensors)
        _case("train", "bf16", 4, 512, 8192),
        # one sequence at the longest length: one GPU's share of the largest problem
        _case("train", "bf16", 1, 1024, 65536),
        # the largest problem: batch 8 at the longest length, 1 GiB tensors
        _case("train", "bf16", 8, 1024, 65536),
        # many short rows in fp32 (262144 of them)
        _case("train", "f32", 64, 4096, 256),
        # a channel-last layer of a language model: 8 sequences of 2048 steps, width 1024
        _case("cl_train", "bf16", 8, 1024, 2048),
        # the same with sizes that are not round: 3 sequences of 1000 steps, width 776
        _case("cl_train", "f16", 3, 776, 1000),
        # one long channel-last sequence
        _case("cl_train", "bf16", 1, 1024, 65536),
        # a layer whose decays come from softplus(z), made inside the scan
        _case("softplus_train", "bf16", 4, 1024, 4096),
        # the contraction scan at a length of several chunks
        _case("dimwise", "f32", 4, 512, 8192),
    ]
    for c in cases:
        c["name"] = "{op}_{dtype}_b{batch}_d{dim}_l{seqlen}".format(**c)
    return cases


def draw(rng):
    op = rng.choice(["fwd", "rev", "train", "train", "train", "cl_fwd", "cl_train", "cl_train",
                     "softplus_fwd", "softplus_train", "dimwise"])
    dtype = rng.choice(["f32", "f16", "bf16"])
    # elements of one tensor, 2^14 .. 2^28, spread over the logarithm
    elements = 2.0 ** rng.uniform(14, 28)
    batch = round(2.0 ** rng.uniform(0, 6))
    if op.startswith("cl_"):
        vec = 16 // SIZE[dtype]
        dim = vec * max(1, round(2.0 ** rng.uniform(5, 12) / vec))
        seqlen = max(1, min(65536, round(elements / (batch * dim))))
    else:
        seqlen = 2 ** rng.randint(6 if op == "dimwise" else 5, 16)
        batch = min(batch, max(1, int(elements / seqlen)))
        dim = max(1, min(8192, round(elements / (batch * seqlen))))
    return _case(op, dtype, batch, dim, seqlen)


# ------------------------------------------------------------------------------ inputs
def _inputs(case, seed):
    """The case's tensors by name, from the seed alone."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    dtype = DTYPES[case["dtype"]]
    B, D, L = case["batch"], case["dim"], case["seqlen"]
    last = case["op"].startswith("cl_")
    shape = (B, L, D) if last else (B, D, L)

    def randn():
        return torch.randn(shape, generator=gen, device="cuda")

    if case["op"] == "dimwise":
        G = fpscan_amd.dimwise_groups(L)
        ax = 0.99 + 0.01 * torch.rand(shape, generator=gen, device="cuda")
        bh = torch.randn((B, D, G), generator=gen, device="cuda") / G
        wq, wk = 0.01 * torch.rand((2, D), generator=gen, device="cuda")
        return {"ax": ax.to(dtype), "bx": (randn() / G).to(dtype), "bh": bh.to(dtype),
                "wq": wq.to(dtype), "wk": wk.to(dtype)}
    rate = 0.001 + 0.099 * torch.rand(D, generator=gen, device="cuda")
    z = randn()
    got = {}
    if case["op"].startswith("softplus"):
        got["z"], got["rate"] = z.to(dtype), rate
    else:
        softplus = torch.nn.functional.softplus(z)
        got["gates"] = torch.exp(-softplus * (rate if last else rate[:, None])).to(dtype)
        del softplus
    del z
    got["tokens"] = (0.1 * randn()).to(dtype)
    if case["op"].endswith("train"):
        got["grad_out"] = randn().to(dtype)
    return got


def prepare(case, seed):
    state = _inputs(case, seed)
    if case["op"].endswith("train"):
        for name in ("gates", "z", "rate", "tokens"):
            if name in state:
                state[name].requires_grad_()
    state["op"] = case["op"]
    return state


# -------------------------------------------------------------------------------- pass
def run(state):
    op = state["op"]
    if op == "fwd":
        return fpscan_amd.scan_forward(state["gates"], state["tokens"])
    if op == "rev":
        return fpscan_amd.scan_forward(state["gates"], state["tokens"], reverse=True)
    if op == "cl_fwd":
        return fpscan_amd.scan_forward_channel_last(state["gates"], state["tokens"])
    if op == "softplus_fwd":
        return fpscan_amd.scan_forward_softplus(state["z"], state["rate"], state["tokens"])
    if op == "dimwise":
        bx = state["bx"].clone()
        fpscan_amd.dimwise_forward(state["ax"], bx, state["bh"], state["wq"], state["wk"])
        return bx
    if op == "softplus_train":
        leaves = (state["z"], state["rate"], state["tokens"])
        out = fpscan_amd.pscan_softplus(*leaves)
    else:
        leaves = (state["gates"], state["tokens"])
        out = (fpscan_amd.pscan_channel_last if op == "cl_train" else fpscan_amd.pscan)(*leaves)
    return (out, *torch.autograd.grad(out, leaves, state["grad_out"]))


# ------------------------------------------------------------------------ bytes, limits
def work(case):
    """Bytes and operations of one pass. A training step is two calls with the loss between
    them: the forward reads two tensors and writes one, the backward reads three and writes
    two."""
    n = case["batch"] * case["dim"] * case["seqlen"]
    train = case["op"].endswith("train")
    return {"bytes": (8 if train else 3) * n * SIZE[case["dtype"]], "flops": (5 if train else 2) * n}


def tolerance(case):
    # about four times the error against 64 bits that these ranges show: one rounding of the
    # output to the type and two in the gradients, which use the rounded output (2.4e-3 in
    # bf16, 3e-4 in f16); in fp32 the sums' own rounding (4e-7; 1.2e-6 with the softplus gates)
    if case["dtype"] == "f32":
        return {"rel": 5e-6 if case["op"].startswith("softplus") else 2e-6, "max": 5e-5}
    return {"rel": 1e-2, "max": 3e-2} if case["dtype"] == "bf16" else {"rel": 1.2e-3, "max": 4e-3}


# ------------------------------------------------------------------- results in 64 bits
def _scan(a, b):
    """y[t] = a[t] y[t-1] + b[t] along the last axis (a[0] is not used), by doubling spans."""
    a, b, L, step = a.clone(), b.clone(), b.shape[-1], 1
    while step < L:
        b[..., step:] += a[..., step:] * b[..., :-step].clone()
        a[..., step:] *= a[..., :-step].clone()
        step *= 2
    return b


def _by_rows(fn, n_out, *tensors):
    """fn over pieces of the leading axis (float64 in, tuples out), put together again."""
    rows = tensors[0].shape[0]
    piece = max(1, (1 << 26) // tensors[0].shape[-1])
    outs = None
    for r in range(0, rows, piece):
        got = fn(*(t[r:r + piece].double() for t in tensors))
        if outs is None:
            outs = [torch.empty((rows,) + g.shape[1:], dtype=torch.float64, device=g.device)
                    for g in got[:n_out]]
        for o, g in zip(outs, got):
            o[r:r + piece] = g
    return outs


def _gradients(a, y, go):
    """(grad_gates, grad_tokens) of a scan with gates a and output y."""
    after = torch.ones_like(a)
    after[..., :-1] = a[..., 1:]
    gx = _scan(after.flip(-1), go.flip(-1)).flip(-1)
    before = torch.zeros_like(y)
    before[..., 1:] = y[..., :-1]
    return gx * before, gx


def _dimwise(case, s):
    """The contraction scan; the scores that pick a group are rounded to the tensors' type."""
    dtype = DTYPES[case["dtype"]]
    L = case["seqlen"]
    W, P = DIMWISE_CHUNK[L]
    C = L // (W * P)
    rows = case["batch"] * case["dim"]

    def rnd(t):
        return t if case["dtype"] == "f32" else t.to(dtype).double()

    per_row = [s[n].double().repeat(case["batch"])[:, None] for n in ("wq", "wk")]

    def piece(ax, bx, bh, wq, wk):
        n = ax.shape[0]
        a = ax.view(n, C, W, P).clone()
        a[:, 0, 0, 0] = 1.0
        local = _scan(a, bx.view(n, C, W, P))
        k = rnd(rnd(wk * bh[:, :W]) + bh[:, :W])
        carry = torch.zeros(n, dtype=torch.float64, device=ax.device)
        for c in range(C):
            y = local[:, c]
            y[:, 0] += a[:, c, 0].cumprod(-1) * carry[:, None]
            v = y[:, :, -1]
            rv = rnd(v)
            q = rnd(rnd(wq * rv) + rv)
            r = v.clone()
            for g in range(1, W - 1):
                score = rnd(k[:, :g] * q[:, g:g + 1])
                m = score.argmax(-1, keepdim=True)
                # the first of the largest
                m = (score == score.gather(1, m)).to(torch.int8).argmax(-1, keepdim=True)
                r[:, g] = (score.gather(1, m) * v.gather(1, m))[:, 0] + v[:, g]
            y[:, 1:] += r[:, :-1, None]
            carry = y[:, -1, -1].clone()
        return (local.reshape(n, L),)

    flat = [s[n].reshape(rows, -1) for n in ("ax", "bx", "bh")]
    return _by_rows(piece, 1, *flat, *per_row)[0].view(case["batch"], case["dim"], L)


def exact(case, seed):
    s = _inputs(case, seed)
    B, D, L, op = case["batch"], case["dim"], case["seqlen"], case["op"]
    if op == "dimwise":
        return _dimwise(case, s)
    last = op.startswith("cl_")

    def rows(t):
        return (t.transpose(1, 2) if last else t).reshape(B * D, L)

    def back(t):
        t = t.view(B, D, L)
        return t.transpose(1, 2).contiguous() if last else t

    x = rows(s["tokens"])
    if op in ("fwd", "cl_fwd"):
        return back(_by_rows(lambda a, b: (_scan(a, b),), 1, rows(s["gates"]), x)[0])
    if op == "rev":
        return back(_by_rows(lambda a, b: (_scan(a.flip(-1), b.flip(-1)).flip(-1),), 1,
                             rows(s["gates"]), x)[0])
    if op in ("train", "cl_train"):
        def step(a, b, go):
            y = _scan(a, b)
            return (y, *_gradients(a, y, go))

        return tuple(back(t) for t in _by_rows(step, 3, rows(s["gates"]), x,
                                               rows(s["grad_out"])))

    def decays(z, rate):
        # softplus without torch's threshold, above which it returns z itself
        sp = z.clamp(min=0) + torch.log1p(torch.exp(-z.abs()))
        return sp, torch.exp(-sp * rate)

    z = rows(s["z"])
    rate = s["rate"].double().repeat(B)[:, None]
    if op == "softplus_fwd":
        return back(_by_rows(lambda z, r, b: (_scan(decays(z, r)[1], b),), 1, z, rate, x)[0])

    def step(z, r, b, go):
        sp, a = decays(z, r)
        y = _scan(a, b)
        ga, gx = _gradients(a, y, go)
        return y, -ga * a * r * torch.sigmoid(z), gx, -(ga * a * sp).sum(-1, keepdim=True)

    y, gz, gx, gr = _by_rows(step, 4, z, rate, x, rows(s["grad_out"]))
    return back(y), back(gz), gr.view(B, D).sum(0), back(gx)
