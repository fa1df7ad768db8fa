"""Mamba3SisoFn for a few tokens (Mamba3StepKernel: the state through registers
in one launch) on the GPU vs the fp64 oracle: key counts at the edges of the
64-key groups and of a four-key group, state rows cut by a row block, the three
row-block heights, one to sixteen tokens (prepared four at a time), angles of
some pairs, Q/K heads shared, with and without Z, D, input and final states,
agreement with the chunked kernel, what lies behind a sequence's tokens, and
outputs over inputs: final states over the
input states (one row block a head), y over V, Z, Q and a part of V."""

import numpy as np
import pytest

import xmetai_onnx_plugins as xp
from oracle import cref
from parity import TOL_GPU, TOL_M3, check, to_dev
from xmetai_onnx_plugins import workloads as W

pytestmark = pytest.mark.gpu

KEYS = ("Q", "K", "V", "ADT", "DT", "Trap", "Q_bias", "K_bias", "Angles", "D", "Z")
STATES = ("ssm", "angle", "k", "v")
S = W.Mamba3SisoShape


def run(s, seed, start=True):
    inp = W.mamba3_siso_inputs(s, seed=seed)
    rng = np.random.default_rng(seed + 1000)
    states = None
    if start:
        states = (rng.standard_normal((s.batch, s.nheads, s.headdim, s.dstate)).astype(np.float32),
                  rng.uniform(0, 2 * np.pi, (s.batch, s.nheads, s.a)).astype(np.float32),
                  rng.standard_normal((s.batch, s.nheads, s.dstate)).astype(np.float32),
                  rng.standard_normal((s.batch, s.nheads, s.headdim)).astype(np.float32))
    y, f = xp.mamba3_siso_fn(*(to_dev(inp[k]) for k in KEYS), return_final_states=True,
                             input_states=tuple(to_dev(x) for x in states) if start else None)
    ref_y, ref_f = cref.mamba3_siso(*(inp[k] for k in KEYS), dtype=np.float64, input_states=states, return_state=True)
    return (y, *f), (ref_y, *ref_f)


def compare(name, got, ref, tol):
    # an angle next to the wrap may come out one period off: compare on the circle
    for part, g, r in zip(("y", *STATES), got, ref):
        g = g.cpu().numpy() if hasattr(g, "cpu") else g
        r = r.cpu().numpy() if hasattr(r, "cpu") else r
        if part == "angle":
            period = 2.0 * float(np.float32(np.pi))
            d = (g.astype(np.float64) - r + period / 2) % period - period / 2
            g = r + d
        check(f"mamba3_siso_step/{name}/{part}", g, r, tol)


def step_rows():
    names = xp.last_launches()
    if len(names) != 1 or not names[0].startswith("Mamba3StepKernel<"):
        return 0
    return 16 * int(names[0][:-1].split(",")[1])


@pytest.mark.parametrize("n", [2, 6, 62, 64, 66, 128, 130, 190, 192, 194, 254, 256])
@pytest.mark.parametrize("tokens", [1, 5])
def test_step_keys(n, tokens):
    got, ref = run(S(2, tokens, 4, 20, n, nheads_qk=2, has_z=True), seed=n)
    assert step_rows() == 16, xp.last_launches()
    compare(f"n{n}_t{tokens}", got, ref, TOL_M3)


@pytest.mark.parametrize("p", [1, 15, 16, 17, 31, 33, 63, 64, 65, 100])
@pytest.mark.parametrize("heads,rows", [(2, 16), (64, 32), (256, 64)])
def test_step_rows(p, heads, rows):
    got, ref = run(S(2, 3, heads, p, 32, angles=5), seed=p)
    assert step_rows() == rows, xp.last_launches()
    compare(f"p{p}_h{heads}", got, ref, TOL_M3)


@pytest.mark.parametrize("p,heads,rows", [(64, 127, 16), (64, 128, 32), (65, 63, 16), (65, 64, 32), (64, 511, 32), (64, 512, 64),
                                          (100, 255, 32), (100, 256, 64)])
def test_step_row_thresholds(p, heads, rows):
    """32 rows from 128 blocks of 64 rows on, 64 from 512."""
    got, ref = run(S(1, 2, heads, p, 32, angles=5), seed=heads)
    assert step_rows() == rows, xp.last_launches()
    compare(f"threshold_p{p}_h{heads}", got, ref, TOL_M3)


@pytest.mark.parametrize("tokens", [1, 2, 4, 7, 8])
@pytest.mark.parametrize("has_z,has_d,start", [(True, True, True), (False, False, True), (True, False, False)])
def test_step_tokens(tokens, has_z, has_d, start):
    got, ref = run(S(2, tokens, 3, 64, 128, angles=40, has_z=has_z, has_d=has_d), seed=tokens, start=start)
    assert step_rows() == 16
    compare(f"t{tokens}_{has_z}_{has_d}_{start}", got, ref, TOL_M3)


@pytest.mark.parametrize("tokens,heads,step", [(9, 128, True), (16, 128, True), (17, 128, False), (9, 4, False)])
def test_step_token_limits(tokens, heads, step):
    got, ref = run(S(2, tokens, heads, 24, 64, has_z=True), seed=tokens)
    assert (step_rows() > 0) == step, xp.last_launches()
    compare(f"limit_t{tokens}_h{heads}", got, ref, TOL_M3)


def test_step_agrees_with_the_chunked_kernel(override):
    s = S(3, 6, 4, 64, 128, has_z=True)
    got, _ = run(s, seed=5)
    assert step_rows() == 16
    override("m3_path", 2)
    chunked, _ = run(s, seed=5)
    assert xp.last_launches() == ["Mamba3ChunkKernel<2,4,8,0>"], xp.last_launches()
    compare("vs_chunked", got, [x.cpu().numpy() for x in chunked], TOL_GPU)


def call_states(dev, states, outs):
    """xm_mamba3_siso_forward_states on device tensors; outs: y and the four states."""
    import ctypes
    import torch
    from xmetai_onnx_plugins import _capi
    ins = [*dev, *states]
    arr = (_capi.XmTensor * len(ins))(*[xp._desc_from_tensor(x) for x in ins])
    attrs = xp._attrs("mamba3_siso", has_d=1, has_z=int(dev[10] is not None), return_final_states=1, has_input_states=1)
    err = ctypes.create_string_buffer(256)
    st = xp.lib().xm_mamba3_siso_forward_states(arr, len(ins), ctypes.byref(attrs), *(x.data_ptr() for x in outs),
                                                torch.cuda.current_stream().cuda_stream, None, err, len(err))
    assert st == xp.XM_OK, err.value
    torch.cuda.synchronize()


def sharing_case(s, seed):
    """Inputs and input states on the device, and the call's results in buffers of their own."""
    import torch
    inp = W.mamba3_siso_inputs(s, seed=seed)
    g = torch.Generator(device="cuda").manual_seed(seed)
    states = [torch.randn((s.batch, s.nheads, *d), generator=g, device="cuda")
              for d in ((s.headdim, s.dstate), (s.a,), (s.dstate,), (s.headdim,))]
    states[1] = states[1].abs()
    dev = [to_dev(inp[k]) for k in KEYS]
    y, f = xp.mamba3_siso_fn(*dev, return_final_states=True, input_states=tuple(states))
    return dev, states, [y, *f]


@pytest.mark.parametrize("tokens", [1, 6, 16])
@pytest.mark.parametrize("p,heads,rows", [(8, 4, 16), (32, 4, 32), (33, 4, 64), (64, 4, 64), (64, 80, 64), (96, 4, 0)])
def test_step_states_in_place(p, heads, rows, tokens):
    """A decode loop may keep one set of state buffers.  Row block 0 writes the k
    and angle states that every row block of a head reads, so a head is one block
    up to 64 rows, and the call the chunked kernel's above (there only ssm and v in place)."""
    import torch
    dev, states, want = sharing_case(S(2, tokens, heads, p, 128, angles=40, has_z=True), seed=p + tokens)
    if p <= 64:
        outs = [torch.empty_like(want[0]), *states]
        call_states(dev, states, outs)
        # 16 tokens of few blocks are the chunked kernel's, whose workgroups of 32 rows own a head of up to 32
        chunked = tokens > 8 and p <= 32
        assert step_rows() == (0 if chunked else rows), xp.last_launches()
    else:
        outs = [torch.empty_like(want[0]), states[0], want[2].clone(), want[3].clone(), states[3]]
        call_states(dev, states, outs)
        assert (step_rows() == 16) == (tokens <= 8), xp.last_launches()
    compare(f"in_place_p{p}_h{heads}_t{tokens}", outs, [x.cpu().numpy() for x in want], TOL_GPU)


@pytest.mark.parametrize("tokens", [1, 4, 5])
@pytest.mark.parametrize("over", ["V", "Z", "Q", "behind_V"])
def test_y_over_an_input(over, tokens):
    """y over V or Z, which a block reads only in its own rows and tokens: as ever;
    over Q, or a part of V: only while a call's tokens are read at once (four)."""
    import torch
    dev, states, want = sharing_case(S(2, tokens, 3, 32, 32, has_z=True), seed=tokens)
    n, row = want[0].numel(), want[0][0, 0].numel()
    if over == "behind_V":   # y one token row before V
        buf = torch.empty(n + row, device="cuda")
        y, v = buf[:n].view(want[0].shape), buf[row:].view(want[0].shape)
        v.copy_(dev[2])
        dev[2] = v
    else:
        y = dev[KEYS.index(over)]
    outs = [y, *(torch.empty_like(x) for x in want[1:])]
    call_states(dev, states, outs)
    assert step_rows() == (0 if over in ("Q", "behind_V") and tokens > 4 else 32 if over == "Q" else 16), xp.last_launches()
    compare(f"y_over_{over}_t{tokens}", outs, [x.cpu().numpy() for x in want], TOL_GPU)


@pytest.mark.parametrize("has_z", [True, False])
@pytest.mark.parametrize("tokens", [1, 2, 3, 5, 6, 7])
def test_step_reads_nothing_behind_its_tokens(tokens, has_z):
    """A block takes four tokens: those past the end read as zeros, whatever
    follows a sequence's rows (here NaN, in the same allocation)."""
    import torch
    s = S(3, tokens, 4, 24, 64, angles=20, has_z=has_z)
    dev, states, want = sharing_case(s, seed=tokens)

    def guarded(x):
        buf = torch.full((x.numel() + 16 * s.nheads * 64,), float("nan"), device="cuda")
        t = buf[:x.numel()].view(x.shape)
        t.copy_(x)
        return t
    outs = [torch.empty_like(x) for x in want]
    call_states([x if x is None else guarded(x) for x in dev], states, outs)
    assert step_rows() == 16
    for g, w in zip(outs, want):
        assert torch.isfinite(g).all() and torch.equal(g, w)
    for b in (1, 2):   # the sequence behind one whose results must not change
        part = [x if x is None else x.clone() for x in dev]
        for i in (0, 1, 2, 3, 4, 5, 8, 10):
            if part[i] is not None:
                part[i][b] = float("nan")
        call_states(part, states, outs)
        for g, w in zip(outs, want):
            assert torch.equal(g[:b], w[:b])
