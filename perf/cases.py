"""The work that callers of the recurrent operators have them do, as timed cases.

Each case is one call of ``selective_scan_fn``, ``gated_deltanet2_fn`` or
``mamba3_siso_fn`` on inputs resident in GPU memory, of the sizes that layers
of language models have: whole batches of training-length rows, one prompt at
a time (prefill), several prompts packed in one row, and single tokens of many
running sequences (decode, state in and state out).  Values follow the
distributions of ``xmetai_onnx_plugins.workloads``.

A decode step goes through a handle built once (``prepare=True``), as a serving
loop keeps one per layer; every other call is the plain function, which
allocates its output.
"""

import math
import os
import sys

import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
_PKG = os.path.join(_ROOT, "xmetai-onnx-plugins_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

_TYPES = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}


def _ss(name, batch, dim, seqlen, dstate, dtype="f32", groups=1, state=False):
    c = dict(op="selective_scan", batch=batch, dim=dim, seqlen=seqlen, dstate=dstate, dtype=dtype, groups=groups,
             state=state)
    return dict(c, name=name) if name else c


def _gdn(name, batch, seqlen, heads, dk, dv, per_key=True, start=True, state=True, packed=0, handle=False):
    c = dict(op="gated_deltanet2", batch=batch, seqlen=seqlen, heads=heads, dk=dk, dv=dv, per_key=per_key, start=start,
             state=state, packed=packed, handle=handle)
    return dict(c, name=name) if name else c


def _m3(name, batch, seqlen, heads, p, n, heads_qk=0, gate=True, start=False, state=True, packed=0, handle=False):
    c = dict(op="mamba3_siso", batch=batch, seqlen=seqlen, heads=heads, p=p, n=n, heads_qk=heads_qk or heads, gate=gate,
             start=start, state=state, packed=packed, handle=handle)
    return dict(c, name=name) if name else c


def listed():
    return [
        # The smallest call in use: the repository's CPU-sized configuration, where latency counts.
        _ss("ss_small", 1, 256, 512, 16),
        # A whole batch through one layer of a 2.8 B model: the benchmark's headline workload.
        _ss("ss_layer", 8, 5120, 2048, 16),
        # One prompt through the same layer, of a length that is no multiple of anything; the state is kept.
        _ss("ss_prompt", 1, 5120, 1999, 16, state=True),
        # Two long prompts in bfloat16.
        _ss("ss_bf16", 2, 4096, 4096, 16, dtype="bf16"),
        # A whole batch, gates equal over the keys of a head: the benchmark's configuration.
        _gdn("gdn2_layer", 4, 4096, 16, 128, 128, per_key=False, state=False),
        # One long document, wide heads, few of them.
        _gdn("gdn2_long", 1, 16384, 8, 256, 256, per_key=False, start=False, state=False),
        # Seven prompts packed in one row, per-key gates; states kept for the decode that follows.
        _gdn("gdn2_packed", 1, 5000, 16, 128, 128, packed=7),
        # One decode step of 32 running sequences, state in and out.
        _gdn("gdn2_decode", 32, 1, 16, 128, 128, handle=True),
        # A whole batch: the benchmark's configuration.
        _m3("m3_layer", 4, 4096, 32, 64, 128, gate=False, state=False),
        # One prompt with the output gate, Q/K shared by head pairs, states kept.
        _m3("m3_prompt", 1, 3001, 32, 64, 128, heads_qk=16),
        # Packed prompts.
        _m3("m3_packed", 1, 4096, 16, 64, 64, packed=5, state=True),
        # One decode step of 32 running sequences.
        _m3("m3_decode", 32, 1, 32, 64, 128, start=True, handle=True),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of these ranges; none has more work than the largest listed case of its operator."""
    kind = rng.choice(["ss", "ss", "gdn", "gdn_packed", "gdn_decode", "m3", "m3_packed", "m3_decode"])
    if kind == "ss":
        dstate = rng.choice([8, 16, 16, 16, 64])
        batch, dim, groups = _log_int(rng, 1, 8), 64 * _log_int(rng, 4, 80), rng.choice([1, 1, 1, 2])
        top = min(4096, 8 * 5120 * 2048 * 16 // (batch * dim * dstate))
        return _ss(None, batch, dim, _log_int(rng, 64, max(64, top)), dstate, dtype=rng.choice(["f32", "f32", "bf16", "f16"]),
                   groups=groups, state=rng.random() < 0.5)
    if kind.startswith("gdn"):
        dk, dv = rng.choice([(64, 64), (128, 128), (128, 128), (128, 65), (192, 128), (256, 256), (320, 64)])
        if kind == "gdn_decode":
            return _gdn(None, _log_int(rng, 1, 64), rng.choice([1, 1, 1, 2, 4]), rng.choice([4, 8, 16]), dk, dv,
                        per_key=rng.random() < 0.5, handle=True)
        heads = rng.choice([4, 8, 16])
        batch = 1 if kind == "gdn_packed" else _log_int(rng, 1, 8)
        top = min(8192, 4 * 4096 * 16 * 128 * 128 // (batch * heads * dk * dv))
        seqlen = _log_int(rng, 48, max(48, top))
        return _gdn(None, batch, seqlen, heads, dk, dv, per_key=rng.random() < 0.5, start=rng.random() < 0.5,
                    state=rng.random() < 0.5, packed=rng.randint(2, 9) if kind == "gdn_packed" else 0)
    p, n, heads = rng.choice([64, 64, 128]), rng.choice([64, 128, 128, 256]), rng.choice([8, 16, 32])
    heads_qk, gate = heads // rng.choice([1, 1, 2, 4]), rng.random() < 0.5
    if kind == "m3_decode":
        return _m3(None, _log_int(rng, 1, 64), rng.choice([1, 1, 1, 2, 4]), heads, p, n, heads_qk=heads_qk, gate=gate,
                   start=True, handle=True)
    batch = 1 if kind == "m3_packed" else _log_int(rng, 1, 8)
    top = min(4096, 4 * 4096 * 32 * 64 * 128 // (batch * heads * p * n))
    return _m3(None, batch, _log_int(rng, 48, max(48, top)), heads, p, n, heads_qk=heads_qk, gate=gate,
               start=rng.random() < 0.5, state=rng.random() < 0.5, packed=rng.randint(2, 9) if kind == "m3_packed" else 0)


# --- inputs ----------------------------------------------------------------

def _offsets(case, seed):
    """Token offsets of the packed sequences: ragged lengths that sum to the row's."""
    if not case["packed"]:
        return None
    g = torch.Generator().manual_seed(seed * 7 + 1)
    cut = torch.randperm(case["seqlen"] - 1, generator=g)[:case["packed"] - 1] + 1
    return [0] + sorted(int(x) for x in cut) + [case["seqlen"]]


def _inputs(case, seed):
    """The operator's input tensors by name, on the GPU, from the seed alone."""
    dev = torch.device("cuda")
    g = torch.Generator(device=dev).manual_seed(seed)

    def normal(*shape):
        return torch.randn(*shape, generator=g, device=dev)

    def uniform(lo, hi, *shape):
        return torch.rand(*shape, generator=g, device=dev) * (hi - lo) + lo

    softplus = torch.nn.functional.softplus
    if case["op"] == "selective_scan":
        b, d, l, n, grp = case["batch"], case["dim"], case["seqlen"], case["dstate"], case["groups"]
        t = _TYPES[case["dtype"]]
        bc = (b, n, l) if grp == 1 else (b, grp, n, l)
        return dict(u=normal(b, d, l).to(t), delta=normal(b, d, l).to(t),
                    A=-torch.exp(uniform(0.0, math.log(16.0), d, n)), B=normal(*bc).to(t), C=normal(*bc).to(t),
                    D=normal(d), delta_bias=uniform(-4.0, -2.0, d))
    offsets = _offsets(case, seed)
    b, t, h = case["batch"], case["seqlen"], case["heads"]
    rows = len(offsets) - 1 if offsets else b
    if case["op"] == "gated_deltanet2":
        k, v = case["dk"], case["dv"]
        i = dict(q=normal(b, t, h, k), k=normal(b, t, h, k), v=normal(b, t, h, v))
        gate = (b, t, h, k if case["per_key"] else 1)
        i["g"] = (-softplus(normal(*gate))).expand(b, t, h, k).contiguous()
        i["beta"] = torch.sigmoid(normal(*gate)).expand(b, t, h, k).contiguous()
        i["w"] = torch.sigmoid(normal(b, t, h, v))
        if case["start"]:
            i["initial_state"] = 0.05 * normal(rows, h, k, v)
    else:
        p, n, hq = case["p"], case["n"], case["heads_qk"]
        rs = 1.0 / math.sqrt(n)
        i = dict(Q=normal(b, t, hq, n) * rs, K=normal(b, t, hq, n) * rs, V=normal(b, t, h, p))
        i["DT"] = softplus(normal(b, h, t) + uniform(-4.0, -2.0, h)[None, :, None])
        i["ADT"] = -torch.exp(uniform(0.0, math.log(16.0), h))[None, :, None] * i["DT"]
        i["Trap"] = uniform(0.0, 1.0, b, h, t)
        i["Q_bias"], i["K_bias"] = normal(h, n) * rs, normal(h, n) * rs
        i["Angles"] = uniform(0.0, 1.0, b, t, h, n // 2)
        i["D"] = normal(h)
        if case["gate"]:
            i["Z"] = normal(b, t, h, p)
        if case["start"]:
            i["input_states"] = (0.1 * normal(rows, h, p, n), uniform(0.0, 2.0 * math.pi, rows, h, n // 2),
                                 normal(rows, h, n) * rs, normal(rows, h, p))
    if offsets:
        i["cu_seqlens"] = torch.tensor(offsets, dtype=torch.int64, device=dev)
    return i


def _call(case, i, prepare=False):
    import xmetai_onnx_plugins as xp
    if case["op"] == "selective_scan":
        return xp.selective_scan_fn(i["u"], i["delta"], i["A"], i["B"], i["C"], i["D"], None, i["delta_bias"],
                                    delta_softplus=True, return_last_state=case["state"], prepare=prepare)
    if case["op"] == "gated_deltanet2":
        return xp.gated_deltanet2_fn(i["q"], i["k"], i["v"], i["g"], i["beta"], i["w"], i.get("initial_state"),
                                     scale=1.0 / math.sqrt(case["dk"]), output_final_state=case["state"],
                                     cu_seqlens=i.get("cu_seqlens"), prepare=prepare)
    return xp.mamba3_siso_fn(i["Q"], i["K"], i["V"], i["ADT"], i["DT"], i["Trap"], i["Q_bias"], i["K_bias"], i["Angles"],
                             i["D"], i.get("Z"), input_states=i.get("input_states"), return_final_states=case["state"],
                             cu_seqlens=i.get("cu_seqlens"), prepare=prepare)


def prepare(case, seed):
    i = _inputs(case, seed)
    return (case, i, _call(case, i, prepare=True) if case.get("handle") else None)


def run(state):
    case, i, handle = state
    return handle() if handle is not None else _call(case, i)


# --- what a pass cannot do without -----------------------------------------

def work(case):
    """Bytes: inputs read once and outputs written once.  Operations: those of the token-by-token recurrence."""
    b = case["batch"]
    if case["op"] == "selective_scan":
        d, l, n = case["dim"], case["seqlen"], case["dstate"]
        size = 4 if case["dtype"] == "f32" else 2
        nbytes = size * (3 * b * d * l + 2 * b * case["groups"] * n * l) + 4 * (d * n + 2 * d)
        nbytes += 4 * b * d * n * case["state"]
        return {"bytes": nbytes, "flops": 7 * b * d * l * n}   # decay exponent and exp2, input, two fused adds
    t, h = case["seqlen"], case["heads"]
    rows = case["packed"] or b
    if case["op"] == "gated_deltanet2":
        k, v = case["dk"], case["dv"]
        nbytes = 4 * b * t * h * (4 * k + 3 * v) + 4 * rows * h * k * v * (case["start"] + case["state"])
        return {"bytes": nbytes, "flops": 7 * b * t * h * k * v}   # decay, erase, write, read
    p, n, a = case["p"], case["n"], case["n"] // 2
    one_state = h * (p * n + a + n + p)
    nbytes = 4 * (2 * b * t * case["heads_qk"] * n + (3 if case["gate"] else 2) * b * t * h * p + b * t * h * a
                  + 3 * b * h * t + 2 * h * n + h + rows * one_state * (case["start"] + case["state"]))
    return {"bytes": nbytes, "flops": 5 * b * t * h * p * n}   # decay, read, write


def tolerance(case):
    """fp32 sums in another order differ by about 1e-6 of the result; 16-bit results by some of their last bits."""
    if case.get("dtype", "f32") != "f32":
        return {"rel": 2e-3 if case["dtype"] == "bf16" else 3e-4}
    return {"rel": 1e-5}


# --- the same in 64 bits ---------------------------------------------------

def _exact_selective_scan(i):
    u, delta, A, B, C, D, bias = (i[x].double() for x in ("u", "delta", "A", "B", "C", "D", "delta_bias"))
    b, d, l = u.shape
    if B.dim() == 3:
        B, C = B[:, None], C[:, None]
    per = d // B.shape[1]
    dt = torch.nn.functional.softplus(delta + bias[:, None], threshold=20.0)
    y, h = torch.empty_like(u), torch.zeros(b, d, A.shape[1], dtype=torch.float64, device=u.device)
    for t in range(l):
        bt, ct = (x[:, :, :, t].repeat_interleave(per, dim=1) for x in (B, C))
        h = torch.exp(dt[:, :, t, None] * A) * h + bt * (dt[:, :, t] * u[:, :, t])[..., None]
        y[:, :, t] = (ct * h).sum(-1)
    return y + D[:, None] * u, h


def _exact_gated_deltanet2(i, scale, lo, hi, row, start):
    q, k, v, g, beta, w = (i[x][row:row + 1, lo:hi].double() for x in ("q", "k", "v", "g", "beta", "w"))
    q = q * (float(torch.tensor(scale, dtype=torch.float32)) * torch.rsqrt((q * q).sum(-1, keepdim=True) + 1e-6))
    k = k * torch.rsqrt((k * k).sum(-1, keepdim=True) + 1e-6)
    s = start.double().clone()
    o = torch.empty_like(v)
    g, bk = torch.exp(g), beta * k
    for t in range(hi - lo):
        s *= g[:, t, :, :, None]
        write = w[:, t] * v[:, t] - (bk[:, t, :, :, None] * s).sum(-2)
        s += k[:, t, :, :, None] * write[:, :, None, :]
        o[:, t] = (q[:, t, :, :, None] * s).sum(-2)
    return o, s


def _exact_mamba3_siso(i, lo, hi, row, states):
    h = i["V"].shape[2]
    q, k = (i[x][row:row + 1, lo:hi].double().repeat_interleave(h // i[x].shape[2], dim=2) + i[y].double()
            for x, y in (("Q", "Q_bias"), ("K", "K_bias")))
    v, ang = (i[x][row:row + 1, lo:hi].double() for x in ("V", "Angles"))
    adt, dt, trap = (i[x][row:row + 1, :, lo:hi].double() for x in ("ADT", "DT", "Trap"))
    pi = float(torch.tensor(math.pi, dtype=torch.float32))   # the operator's angles turn by a single-precision pi
    gate = torch.sigmoid(trap)
    look = dt * (1.0 - gate)
    weight = dt * gate + torch.cat([look[..., 1:], torch.zeros_like(look[..., :1])], dim=-1)
    if states is None:
        s = torch.zeros(1, h, v.shape[-1], q.shape[-1], dtype=torch.float64, device=v.device)
        theta0 = torch.zeros(1, h, ang.shape[-1], dtype=torch.float64, device=v.device)
    else:
        s, theta0, k_in, v_in = (x[:1].double() for x in states)
        s = s + v_in[..., None] * (k_in * look[..., 0, None])[..., None, :]
    theta = theta0[:, None] + torch.cumsum(torch.tanh(ang) * dt.transpose(1, 2)[..., None] * pi, dim=1)
    theta = theta - 2.0 * pi * torch.floor(theta / (2.0 * pi))
    diag = i["D"].double() + (q * k).sum(-1) * (dt * gate).transpose(1, 2)
    c, sn = torch.cos(theta), torch.sin(theta)

    def turned(x):
        a, b = x[..., 0::2], x[..., 1::2]
        return torch.stack([a * c - b * sn, a * sn + b * c], dim=-1).flatten(-2)

    q, k = turned(q), turned(k)
    decay = torch.exp(adt)
    y = torch.empty_like(v)
    for t in range(hi - lo):
        s = s * decay[:, :, t, None, None]
        y[:, t] = (s * q[:, t, :, None, :]).sum(-1)
        s = s + v[:, t, :, :, None] * (k[:, t] * weight[:, :, t, None])[:, :, None, :]
    y = y + diag[..., None] * v
    if "Z" in i:
        z = i["Z"][row:row + 1, lo:hi].double()
        y = y * z * torch.sigmoid(z)
    return y, (s, theta[:, -1], k[:, -1], v[:, -1])


def exact(case, seed):
    i = _inputs(case, seed)
    if case["op"] == "selective_scan":
        y, h = _exact_selective_scan(i)
        return (y, h) if case["state"] else y
    offsets = _offsets(case, seed)
    parts = [(0, lo, hi) for lo, hi in zip(offsets, offsets[1:])] if offsets else [(r, 0, case["seqlen"])
                                                                               for r in range(case["batch"])]
    outs = []
    for n, (row, lo, hi) in enumerate(parts):
        if case["op"] == "gated_deltanet2":
            shape = (1, case["heads"], case["dk"], case["dv"])
            start = i["initial_state"][n:n + 1] if case["start"] else torch.zeros(shape, device=i["q"].device)
            outs.append(_exact_gated_deltanet2(i, 1.0 / math.sqrt(case["dk"]), lo, hi, row, start))
        else:
            states = tuple(x[n:n + 1] for x in i["input_states"]) if case["start"] else None
            outs.append(_exact_mamba3_siso(i, lo, hi, row, states))
    y = torch.cat([o[0] for o in outs], dim=1 if offsets else 0)
    if not case["state"]:
        return y
    if case["op"] == "gated_deltanet2":
        return y, torch.cat([o[1] for o in outs])
    return y, tuple(torch.cat(x) for x in zip(*(o[1] for o in outs)))
