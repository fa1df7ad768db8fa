"""Mamba3SisoFn's chunked kernel split along the sequence (segments' end states
handed over through the output rows) on the GPU vs the fp64 oracle: every key
tiling, row blocks of 16 and 32 rows and several of them, ragged last segments,
partial angles, shared Q/K heads, with and without Z, D, input and final states,
packed sequences shorter and longer than a segment and empty ones, growth that
overflows a plain decay, infinite and NaN inputs, the automatic choice, and outputs that share memory
with an input, final states over the input states among them (no split)."""

import numpy as np
import pytest

import xmetai_onnx_plugins as xp
from oracle import cref
from parity import Gate, TOL_GPU, TOL_M3, check, to_dev
from xmetai_onnx_plugins import workloads as W

pytestmark = pytest.mark.gpu

KEYS = ("Q", "K", "V", "ADT", "DT", "Trap", "Q_bias", "K_bias", "Angles", "D", "Z")
PARTS = ("y", "ssm", "angle", "k", "v")
S = W.Mamba3SisoShape


def split_launched():
    names = [k.split("<")[0] for k in xp.last_launches() if not k.startswith("PackedGaps")]
    return names == ["Mamba3ChunkKernel", "Mamba3SegCombineKernel", "Mamba3ChunkKernel"]


def start_states(s, n, seed):
    rng = np.random.default_rng(seed)
    return (rng.standard_normal((n, s.nheads, s.headdim, s.dstate)).astype(np.float32),
            rng.uniform(0, 2 * np.pi, (n, s.nheads, s.a)).astype(np.float32),
            rng.standard_normal((n, s.nheads, s.dstate)).astype(np.float32),
            rng.standard_normal((n, s.nheads, s.headdim)).astype(np.float32))


def compare(name, got, ref, tol):
    for part, g, r in zip(PARTS, got, ref):
        g = g.cpu().numpy() if hasattr(g, "cpu") else g
        if part == "angle":   # on the circle: an angle next to the wrap may come out one period off
            period = 2.0 * float(np.float32(np.pi))
            g = r + (g.astype(np.float64) - r + period / 2) % period - period / 2
        check(f"mamba3_siso_split/{name}/{part}", g, r, tol)


CASES = {
    "n64_p64_t600": S(1, 600, 2, 64, 64, has_z=True),
    "n30_p32_t500": S(2, 500, 3, 32, 30),
    "n128_p64_t1000_hq2": S(1, 1000, 4, 64, 128, nheads_qk=2, has_z=True),
    "n128_p16_t900_angles40": S(1, 900, 3, 16, 128, angles=40, has_z=True),
    "n100_p48_t777": S(2, 777, 2, 48, 100),
    "n128_p160_t640": S(1, 640, 2, 160, 128, has_d=False),
    "n192_p64_t1111": S(1, 1111, 2, 64, 192, has_z=True),
    "n256_p80_t1300": S(1, 1300, 2, 80, 256, has_z=True),
    "n64_p64_t2049": S(1, 2049, 1, 64, 64),
}


@pytest.mark.parametrize("name", sorted(CASES))
@pytest.mark.parametrize("start", [True, False])
def test_split_parity(name, start, override):
    s = CASES[name]
    inp = W.mamba3_siso_inputs(s, seed=41)
    states = start_states(s, s.batch, 42) if start else None
    override("m3_split", 2)
    y, f = xp.mamba3_siso_fn(*(to_dev(inp[k]) for k in KEYS), return_final_states=True,
                             input_states=tuple(to_dev(x) for x in states) if start else None)
    assert split_launched(), xp.last_launches()
    ref_y, ref_f = cref.mamba3_siso(*(inp[k] for k in KEYS), dtype=np.float64, input_states=states, return_state=True)
    # hundreds of angle steps: the device within 8 times the reference's own fp32 evaluation (tests/parity.py)
    y32, f32 = cref.mamba3_siso(*(inp[k] for k in KEYS), dtype=np.float32, input_states=states, return_state=True)
    check(f"mamba3_siso_split/{name}/y", y.cpu().numpy(), ref_y, TOL_M3, ref32=y32)
    for part, g, r, r32 in zip(PARTS[1:], f, ref_f, f32):
        if part != "angle":
            check(f"mamba3_siso_split/{name}/{part}", g.cpu().numpy(), r, TOL_M3, ref32=r32)
    override("m3_split", 1)   # the angles with the rest against the whole pass
    y1, f1 = xp.mamba3_siso_fn(*(to_dev(inp[k]) for k in KEYS), return_final_states=True,
                               input_states=tuple(to_dev(x) for x in states) if start else None)
    assert not split_launched()
    compare(f"{name}/vs_whole", (y, *f), [x.cpu().numpy() for x in (y1, *f1)], TOL_GPU)


@pytest.mark.parametrize("offsets", [[0, 700, 1400], [0, 40, 41, 1400], [0, 0, 600, 600, 1400], [3, 500, 1390], [0, 600, 20, 20]])
@pytest.mark.parametrize("start", [True, False])
def test_split_packed(offsets, start, override):
    """Also offsets that fall: [0, 600), nothing, nothing (the device sees that
    they do not rise and keeps the sequences whole)."""
    s = S(1, 1400, 2, 64, 128, has_z=True)
    inp = W.mamba3_siso_inputs(s, seed=43)
    n = len(offsets) - 1
    states = start_states(s, n, 44) if start else None
    cu = to_dev(np.asarray(offsets, np.int64))

    def call():
        y, f = xp.mamba3_siso_fn(*(to_dev(inp[k]) for k in KEYS), return_final_states=True, cu_seqlens=cu,
                                 input_states=tuple(to_dev(x) for x in states) if start else None)
        return (y, *f)
    override("m3_split", 2)
    got = call()
    assert split_launched(), xp.last_launches()
    override("m3_split", 1)
    compare(f"packed_{n}_{start}", got, [x.cpu().numpy() for x in call()], TOL_GPU)


def test_split_growth_beyond_one_decay(override):
    """ADT > 0: a segment grows by exp(128), beyond a float, from a state of 1e-30
    and from none."""
    s = S(1, 800, 2, 32, 64, has_d=False)
    inp = W.mamba3_siso_inputs(s, seed=45)
    inp["ADT"][:] = 0.0
    inp["ADT"][:, :, 300:428] = 1.0
    inp["V"][:, :, :, 1:] = 0.0
    inp["V"][:] *= 1e-30
    inp["V"][:, 200:] = 0.0
    override("m3_split", 2)
    y, f = xp.mamba3_siso_fn(*(to_dev(inp[k]) for k in KEYS), return_final_states=True)
    assert split_launched(), xp.last_launches()
    ref_y, ref_f = cref.mamba3_siso(*(inp[k] for k in KEYS), dtype=np.float64, return_state=True)
    # exp of a sum of 128 instead of 128 factors: 128 x 2^-23 and a few ulp, against factors within 2^-22 each
    # (a row of y holds one value, a sum over the keys that may cancel down to the
    # measure's floor of 1e-3 of the largest: 1e3 times the bound)
    check("mamba3_siso_split/growth/y", y.cpu().numpy(), ref_y, Gate(1e-4, 1e-1))
    check("mamba3_siso_split/growth/ssm", f[0].cpu().numpy(), ref_f[0], 1e-4)


NOT_FINITE = {   # input, place, value
    "v_inf": ("V", (0, 300, 1, 5), np.inf),
    "v_minus_inf_first": ("V", (0, 0, 1, 5), -np.inf),
    "v_nan": ("V", (0, 300, 1, 5), np.nan),
    "k_inf": ("K", (0, 300, 0, 4), np.inf),
    "k_inf_last_of_a_segment": ("K", (0, 223, 0, 7), -np.inf),
    "adt_inf": ("ADT", (0, 1, 300), np.inf),
    "adt_minus_inf": ("ADT", (0, 1, 300), -np.inf),
    "dt_inf": ("DT", (0, 1, 300), np.inf),
    "angle_nan": ("Angles", (0, 300, 1, 2), np.nan),
    "q_inf": ("Q", (0, 300, 0, 4), np.inf),
}


@pytest.mark.parametrize("name", sorted(NOT_FINITE))
@pytest.mark.parametrize("shape,cu", [(S(1, 1000, 2, 64, 64, has_z=True), None), (S(1, 1000, 2, 48, 128, angles=40), None),
                                      (S(1, 1100, 2, 32, 256), [0, 1000, 1100])], ids=["n64", "n128", "n256_packed"])
def test_split_of_infinite_and_nan_inputs(name, shape, cu, override):
    """An infinite or NaN input makes every later state of its rows or heads so, at
    the same places and with the same signs as the whole pass (turning a segment's
    end state would mix infinities of two keys); all else stays as it was."""
    inp = W.mamba3_siso_inputs(shape, seed=51)
    key, at, value = NOT_FINITE[name]
    inp[key][at] = value
    out = []
    for mode in (2, 1):
        override("m3_split", mode)
        y, f = xp.mamba3_siso_fn(*(to_dev(inp[k]) for k in KEYS), return_final_states=True,
                                 cu_seqlens=None if cu is None else to_dev(np.asarray(cu, np.int64)))
        assert split_launched() == (mode == 2), xp.last_launches()
        out.append([x.cpu().numpy() for x in (y, *f)])
    finite = []
    for part, a, b in zip(PARTS, *out):
        np.testing.assert_array_equal(np.where(np.isfinite(a), 0.0, a), np.where(np.isfinite(b), 0.0, b), err_msg=part)
        finite.append((np.where(np.isfinite(a), a, 0.0), np.where(np.isfinite(b), b, 0.0)))
    compare(f"{name}_n{shape.dstate}", *zip(*finite), TOL_GPU)


def test_split_chosen_for_one_prompt():
    s = S(1, 1001, 32, 64, 128, has_z=True)
    inp = W.mamba3_siso_inputs(s, seed=46)
    y = xp.mamba3_siso_fn(*(to_dev(inp[k]) for k in KEYS))
    assert split_launched(), xp.last_launches()
    check("mamba3_siso_split/b1_t1001_h32", y.cpu().numpy(), cref.mamba3_siso(*(inp[k] for k in KEYS), dtype=np.float64),
          TOL_M3, ref32=cref.mamba3_siso(*(inp[k] for k in KEYS), dtype=np.float32))


@pytest.mark.parametrize("offsets,heads,split", [([0, 1100, 2000], 8, True), ([0, 40, 2000], 8, True), ([0, 0, 1990], 16, True),
                                                 ([0, 1000, 2000], 17, False), ([0, 90, 200, 310], 2, False)])
def test_split_chosen_for_packed_rows(offsets, heads, split):
    """Packed: up to a quarter of a row block per CU (2 sequences x 16 heads of 64
    rows here), where sequences of even length would gain; each against itself alone."""
    s = S(1, offsets[-1], heads, 64, 64, has_z=True)
    inp = W.mamba3_siso_inputs(s, seed=52)
    n = len(offsets) - 1
    states = [to_dev(x) for x in start_states(s, n, 53)]
    dev = {k: to_dev(inp[k]) for k in KEYS}
    y, f = xp.mamba3_siso_fn(*dev.values(), return_final_states=True, cu_seqlens=to_dev(np.asarray(offsets, np.int64)),
                             input_states=tuple(states))
    assert split_launched() == split, xp.last_launches()
    for b, (lo, hi) in enumerate(zip(offsets, offsets[1:])):
        if lo == hi:
            continue
        part = [x if k in ("Q_bias", "K_bias", "D") else (x[:, :, lo:hi] if k in ("ADT", "DT", "Trap") else x[:, lo:hi]).contiguous()
                for k, x in dev.items()]
        y1, f1 = xp.mamba3_siso_fn(*part, return_final_states=True, input_states=tuple(x[b:b + 1].contiguous() for x in states))
        compare(f"chosen_packed_h{heads}_{b}", (y[:, lo:hi], *(x[b:b + 1] for x in f)), [x.cpu().numpy() for x in (y1, *f1)], TOL_GPU)


def test_output_over_an_input_is_not_split(override):
    import ctypes
    import torch
    from xmetai_onnx_plugins import _capi
    s = S(1, 640, 2, 64, 128)
    inp = W.mamba3_siso_inputs(s, seed=47)
    override("m3_split", 2)
    dev = [to_dev(inp[k]) for k in KEYS]
    want = xp.mamba3_siso_fn(*dev)
    assert split_launched()
    arr = (_capi.XmTensor * len(dev))(*[xp._desc_from_tensor(x) for x in dev])
    attrs = xp._attrs("mamba3_siso", has_d=1, has_z=0)
    err = ctypes.create_string_buffer(256)
    st = xp.lib().xm_mamba3_siso_forward(arr, len(dev), ctypes.byref(attrs), dev[2].data_ptr(),
                                         torch.cuda.current_stream().cuda_stream, None, err, len(err))
    assert st == xp.XM_OK, err.value
    assert not split_launched()
    torch.cuda.synchronize()
    check("mamba3_siso_split/in_place", dev[2].cpu().numpy(), want.cpu().numpy(), TOL_GPU)


def test_overlapping_packed_sequences_keep_their_states(override):
    """Falling offsets may give two sequences the same rows ([0, 900) and [300,
    1400) here); their final states are those of the whole pass."""
    s = S(1, 1400, 2, 64, 128)
    inp = W.mamba3_siso_inputs(s, seed=48)
    cu = to_dev(np.asarray([0, 900, 300, 1400], np.int64))
    out = []
    for mode in (2, 1):
        override("m3_split", mode)
        y, f = xp.mamba3_siso_fn(*(to_dev(inp[k]) for k in KEYS), return_final_states=True, cu_seqlens=cu)
        out.append([x.cpu().numpy() for x in f])
    for part, a, b in zip(PARTS[1:], *out):
        np.testing.assert_array_equal(a, b, err_msg=part)


@pytest.mark.parametrize("p,parts", [(32, (0, 1, 2, 3)), (64, (0, 3)), (64, (0,)), (32, (1,)), (32, (2,)), (64, (3,)), (64, ())])
def test_final_states_over_the_input_states_are_not_split(p, parts):
    """One workgroup walks the whole sequence of its rows and may keep the states
    in one buffer (angle and k up to 32 rows, one workgroup a head); the segments'
    workgroups of one launch may not.  y and the other states apart."""
    import ctypes
    import torch
    from xmetai_onnx_plugins import _capi
    s = S(1, 1001, 4, p, 128, has_z=True)
    inp = W.mamba3_siso_inputs(s, seed=49)
    dev = [to_dev(inp[k]) for k in KEYS]
    states = [to_dev(x) for x in start_states(s, 1, 50)]
    y, f = xp.mamba3_siso_fn(*dev, return_final_states=True, input_states=tuple(states))
    assert split_launched(), xp.last_launches()
    outs = [torch.empty_like(y), *(states[i] if i in parts else torch.empty_like(f[i]) for i in range(4))]
    ins = [*dev, *states]
    arr = (_capi.XmTensor * len(ins))(*[xp._desc_from_tensor(x) for x in ins])
    attrs = xp._attrs("mamba3_siso", has_d=1, has_z=1, return_final_states=1, has_input_states=1)
    err = ctypes.create_string_buffer(256)
    st = xp.lib().xm_mamba3_siso_forward_states(arr, len(ins), ctypes.byref(attrs), *(x.data_ptr() for x in outs),
                                                torch.cuda.current_stream().cuda_stream, None, err, len(err))
    assert st == xp.XM_OK, err.value
    assert split_launched() == (not parts), xp.last_launches()
    torch.cuda.synchronize()
    compare(f"states_in_place_p{p}_{parts}", outs, [x.cpu().numpy() for x in (y, *f)], TOL_GPU)
