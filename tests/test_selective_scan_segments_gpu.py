"""SelectiveScanFn's whole pass run as segments of the sequence (two launches,
the segments' states handed over through the output rows) on the GPU vs the
fp64 oracle, through the C ABI: ragged last tiles and segments, rows on every
4-byte offset, groups, the state layouts, 16-bit rows of even and odd length,
the last state, the automatic choice, growth that overflows a plain decay
product, infinite and NaN inputs, and outputs that share memory with an input (the whole pass), the last
state over A among them."""

import numpy as np
import pytest

from oracle import cref
from parity import TOL_GPU, TOL_SS, check, to_dev
from xmetai_onnx_plugins import last_launches, selective_scan_fn, workloads as W

pytestmark = pytest.mark.gpu

KEYS = ("u", "delta", "A", "B", "C", "D", "z", "delta_bias")
S = W.SelectiveScanShape


def run_ref(inp, state=True):
    return cref.selective_scan(*(inp[k] for k in KEYS[:6]), None, inp["delta_bias"], delta_softplus=True,
                               dtype=np.float64, return_state=state)


def segments_launched():
    # state and output launches of the segmented pass end in mode 1 and 2
    names = [k for k in last_launches() if k.startswith("SelectiveScanFwdKernel")]
    return len(names) == 2 and names[0].endswith(",1>") and names[1].endswith(",2>")


CASES = {
    "n16_l512": S(1, 40, 512, 16),
    "n16_l511_ragged": S(2, 64, 511, 16),
    "n16_l514_short_last": S(1, 32, 514, 16),
    "n16_l1025_groups2": S(1, 128, 1025, 16, groups=2),
    "n3_l900": S(1, 40, 900, 3),
    "n8_l901": S(2, 72, 901, 8),
    "n24_l700": S(1, 33, 700, 24),
    "n64_l1030": S(1, 20, 1030, 64),
    "n100_l1300": S(1, 17, 1300, 100),
    "n256_l1200": S(1, 16, 1200, 256),
}


@pytest.mark.parametrize("name", sorted(CASES))
def test_segments_parity(name, override):
    inp = W.selective_scan_inputs(CASES[name], seed=31)
    override("ss_split", 3)
    y, h = selective_scan_fn(*(to_dev(inp[k]) for k in KEYS), delta_softplus=True, return_last_state=True)
    assert segments_launched(), last_launches()
    ref_y, ref_h = run_ref(inp)
    check(f"selective_scan_segments/{name}/y", y.cpu().numpy(), ref_y, TOL_SS)
    check(f"selective_scan_segments/{name}/h", h.cpu().numpy(), ref_h, TOL_SS)


@pytest.mark.parametrize("split", [1, 2, 3])
@pytest.mark.parametrize("shift", [1, 2, 3])
def test_rows_on_dword_offsets(shift, split, override):
    """u, delta, B, C 4, 8 and 12 bytes off a 16-byte boundary; what follows the
    tensors is infinite and must not reach the last group of their last rows."""
    import torch
    inp = W.selective_scan_inputs(S(1, 64, 517, 16), seed=32)

    def shifted(x):
        buf = torch.full((x.size + 8,), float("inf"), dtype=torch.float32, device="cuda")
        t = buf[shift:shift + x.size].view(x.shape)
        t.copy_(torch.from_numpy(x))
        return t
    override("ss_split", split)
    y = selective_scan_fn(*(shifted(inp[k]) if k in ("u", "delta", "B", "C") else to_dev(inp[k]) for k in KEYS),
                          delta_softplus=True)
    check(f"selective_scan_segments/shift{shift}_{split}", y.cpu().numpy(), run_ref(inp, state=False), TOL_SS)


@pytest.mark.parametrize("fmt", ["float16", "bfloat16"])
@pytest.mark.parametrize("length", [1000, 1002, 1001])   # 8-byte, 4-byte and 2-byte rows
def test_segments_16bit(fmt, length, override):
    """y within one unit of the 16-bit format plus 1e-5 of the oracle on the rounded inputs."""
    import torch
    tdt, mant = getattr(torch, fmt), {"float16": 10, "bfloat16": 7}[fmt]
    inp = W.selective_scan_inputs(S(1, 64, length, 16), seed=33)
    dev = {k: to_dev(x).to(tdt) if k in ("u", "delta", "z", "B", "C") else to_dev(x) for k, x in inp.items()}
    rounded = {k: x.float().cpu().numpy() for k, x in dev.items()}
    override("ss_split", 3)
    y, h = selective_scan_fn(*(dev[k] for k in KEYS), delta_softplus=True, return_last_state=True)
    assert segments_launched(), last_launches()
    ref_y, ref_h = run_ref(rounded)
    got = y.float().cpu().numpy().astype(np.float64)
    spacing = 2.0 ** (np.floor(np.log2(np.maximum(np.abs(ref_y), 2.0 ** -14))) - mant)
    assert np.all(np.abs(got - ref_y) <= spacing + 1e-5)
    check(f"selective_scan_segments_16bit/{fmt}_{length}/h", h.cpu().numpy(), ref_h, TOL_SS)


def test_segments_chosen_for_one_prompt():
    inp = W.selective_scan_inputs(S(1, 5120, 1001, 16), seed=34)
    y = selective_scan_fn(*(to_dev(inp[k]) for k in KEYS), delta_softplus=True)
    assert segments_launched(), last_launches()
    check("selective_scan_segments/b1_d5120_l1001", y.cpu().numpy(), run_ref(inp, state=False), TOL_SS)


@pytest.mark.parametrize("u0", [0.0, 1.0])
def test_growth_beyond_one_decay_product(u0, override):
    """A > 0: a 64-token segment's decay product exp(128) overflows a float
    while the state, zero or 1e-30 before it, stays in range."""
    import torch
    D, N, L = 32, 16, 1024
    dev = torch.device("cuda")
    delta = torch.zeros(1, D, L, device=dev)
    delta[:, :, 0] = 1e-30            # the input of token 0 is 1e-30 u
    delta[:, :, 512:576] = 2.0
    u = torch.zeros(1, D, L, device=dev)
    u[:, :, 0] = u0
    A = torch.ones(D, N, device=dev)
    B = torch.ones(1, N, L, device=dev)
    override("ss_split", 3)
    y = selective_scan_fn(u, delta, A, B, B, None, None, None)
    assert segments_launched(), last_launches()
    want = u0 * 1e-30 * N * np.exp(128.0)
    got = y[0, :, -1].double().cpu().numpy()
    assert np.all(np.abs(got - want) <= 1e-4 * abs(want))   # 64 factors exp2(2 log2 e), each within 4 x 2^-23


NOT_FINITE = {   # input, place, value
    "u_inf": ("u", (0, 3, 300), np.inf),
    "u_nan": ("u", (0, 3, 300), np.nan),
    "u_minus_inf_first": ("u", (0, 3, 0), -np.inf),
    "delta_inf": ("delta", (0, 3, 300), np.inf),
    "b_inf": ("B", (0, 0, 2, 300), np.inf),
    "c_inf": ("C", (0, 0, 2, 300), np.inf),
    "a_inf": ("A", (3, 0), np.inf),
    "a_minus_inf": ("A", (3, 0), -np.inf),
}


@pytest.mark.parametrize("name", sorted(NOT_FINITE))
@pytest.mark.parametrize("shape", [S(1, 64, 1000, 16), S(1, 40, 999, 3), S(2, 64, 1021, 8), S(1, 32, 1100, 64)],
                         ids=["n16", "n3_ragged", "n8", "n64"])
@pytest.mark.parametrize("softplus", [True, False])
def test_infinite_and_nan_inputs(name, shape, softplus, override):
    """Infinite and NaN states (without softplus the states of this input overflow
    by themselves) come out where and as they do in the whole pass."""
    inp = W.selective_scan_inputs(shape, seed=37)
    key, at, value = NOT_FINITE[name]
    inp[key].reshape((shape.batch, 1, shape.dstate, shape.seqlen) if key in "BC" else inp[key].shape)[at] = value
    out = []
    for split in (3, 1):
        override("ss_split", split)
        y, h = selective_scan_fn(*(to_dev(inp[k]) for k in KEYS), delta_softplus=softplus, return_last_state=True)
        assert segments_launched() == (split == 3), last_launches()
        out.append((y.cpu().numpy(), h.cpu().numpy()))
    for part, a, b in zip("yh", *out):
        np.testing.assert_array_equal(np.where(np.isfinite(a), 0.0, a), np.where(np.isfinite(b), 0.0, b), err_msg=part)
        if softplus:   # states of one size: held to the tolerance between two device paths
            check(f"selective_scan_segments/{name}_n{shape.dstate}/{part}", np.where(np.isfinite(a), a, 0.0),
                  np.where(np.isfinite(b), b, 0.0), TOL_GPU)


def test_output_over_an_input_takes_the_whole_pass(override):
    """In place on u, as the C entry point allows: the output rows may not hold records then."""
    import ctypes
    import torch
    import xmetai_onnx_plugins as xp
    from xmetai_onnx_plugins import _capi
    inp = W.selective_scan_inputs(S(1, 64, 512, 16), seed=35)
    override("ss_split", 3)
    dev = [to_dev(inp[k]) for k in KEYS]
    arr = (_capi.XmTensor * len(dev))(*[xp._desc_from_tensor(x) for x in dev])
    attrs = xp._attrs("selective_scan", delta_softplus=1)
    err = ctypes.create_string_buffer(256)
    st = xp.lib().xm_selective_scan_forward(arr, len(dev), ctypes.byref(attrs), dev[0].data_ptr(),
                                            torch.cuda.current_stream().cuda_stream, None, err, len(err))
    assert st == xp.XM_OK, err.value
    assert not segments_launched()
    torch.cuda.synchronize()
    check("selective_scan_segments/in_place", dev[0].cpu().numpy(), run_ref(inp, state=False), TOL_SS)


def test_last_state_over_the_weights_takes_the_whole_pass(override):
    """The last state of one sequence has A's size: over A, whose channel one
    workgroup of the whole pass reads before it writes."""
    import ctypes
    import torch
    import xmetai_onnx_plugins as xp
    from xmetai_onnx_plugins import _capi
    inp = W.selective_scan_inputs(S(1, 64, 512, 16), seed=36)
    override("ss_split", 3)
    dev = [to_dev(inp[k]) for k in KEYS]
    y = torch.empty_like(dev[0])
    arr = (_capi.XmTensor * len(dev))(*[xp._desc_from_tensor(x) for x in dev])
    attrs = xp._attrs("selective_scan", delta_softplus=1, return_last_state=1)
    err = ctypes.create_string_buffer(256)
    st = xp.lib().xm_selective_scan_forward_states(arr, len(dev), ctypes.byref(attrs), y.data_ptr(), dev[2].data_ptr(),
                                                   torch.cuda.current_stream().cuda_stream, None, err, len(err))
    assert st == xp.XM_OK, err.value
    assert not segments_launched(), last_launches()
    torch.cuda.synchronize()
    ref_y, ref_h = run_ref(inp)
    check("selective_scan_segments/last_state_over_A/y", y.cpu().numpy(), ref_y, TOL_SS)
    check("selective_scan_segments/last_state_over_A/h", dev[2].cpu().numpy()[None], ref_h, TOL_SS)
