"""Which kernel a call takes, where an output shares memory with an input above all, read
from xm_last_launches without a GPU: the addresses are made up and nothing runs
(so the file skips itself where a GPU is visible).  The runs on the GPU, for
the cases whose result does not depend on the order of the workgroups, are in the
operators' GPU tests."""

import ctypes

import pytest

import xmetai_onnx_plugins as xp
from xmetai_onnx_plugins import _capi


@pytest.fixture(autouse=True)
def _no_gpu():
    import torch
    if torch.cuda.is_available():
        pytest.skip("made-up addresses: only where no kernel can run")


def launches(op, shapes, outs, at=(), **attrs):
    """Kernels that xm_<op>_forward_states enqueues for inputs of these shapes
    (None: absent) at 1 GiB steps, in order, and then the outputs; `at`: output
    index -> (input index, byte offset) for an output placed over an input."""
    addr = [(i + 1) << 30 for i in range(len(shapes) + outs)]
    ins = (_capi.XmTensor * len(shapes))(*[xp._desc_from_shape(sh, a) if sh is not None else xp._desc_from_tensor(None)
                                           for sh, a in zip(shapes, addr)])
    out = addr[len(shapes):]
    for o, (i, off) in dict(at).items():
        out[o] = addr[i] + off
    a, err = xp._attrs(op, **attrs), ctypes.create_string_buffer(512)
    getattr(xp.lib(), f"xm_{op}_forward_states")(ins, len(shapes), ctypes.byref(a), *out, None, None, err, len(err))
    return [k.split("<")[0] for k in xp.last_launches()]


def m3_launches(b, t, h, p, n, a, at=()):
    qk, th, hn = (b, t, h, n), (b, h, t), (h, n)
    shapes = [qk, qk, (b, t, h, p), th, th, th, hn, hn, (b, t, h, a), (h,), None, (b, h, p, n), (b, h, a), (b, h, n),
              (b, h, p)]
    return launches("mamba3_siso", shapes, 5, at, has_d=1, has_z=0, return_final_states=1, has_input_states=1)


STEP = ["Mamba3StepKernel"]


@pytest.mark.parametrize("t", [1, 4])
@pytest.mark.parametrize("at,one_block", [
    ({}, False),
    ({1: (11, 0)}, False), ({4: (14, 0)}, False),   # ssm and v in place: a row block's own
    ({2: (12, 0)}, True), ({3: (13, 0)}, True),     # angle and k in place
    ({3: (13, 508)}, True), ({3: (13, 512)}, False),   # k over the last value of k, and just behind
    ({3: (1, 0)}, True), ({2: (8, 4)}, True), ({0: (0, 0)}, True), ({1: (9, 0)}, True), ({4: (6, 0)}, True),
], ids=str)
def test_m3_step_with_outputs_over_inputs(at, one_block, t):
    """An output over what all row blocks of a head read: one row block, or (above 64 rows) not this kernel."""
    for p in (16, 32, 64):
        got = m3_launches(1, t, 1, p, 128, 40, at)
        assert got == STEP
        rows = 16 * int(xp.last_launches()[0][:-1].split(",")[1])
        assert rows >= p if one_block else rows == 16
    assert (m3_launches(1, t, 1, 65, 128, 40, at) == STEP) == (not one_block)


def test_m3_step_reads_its_tokens_four_at_a_time():
    row = 32 * 4
    for t, ok in ((4, True), (5, False)):
        assert (m3_launches(1, t, 1, 32, 32, 16, {0: (2, row)}) == STEP) == ok    # y one token behind V
        assert (m3_launches(1, t, 1, 32, 32, 16, {0: (0, 0)}) == STEP) == ok      # y over Q
        assert m3_launches(1, t, 1, 32, 32, 16, {0: (2, 0)}) == STEP              # y over V


def test_ss_segments_with_outputs_over_inputs():
    """y or the last state over an input, or over each other: one launch, not two of segments."""
    u, w, bc = (1, 5120, 2048), (5120, 16), (1, 1, 16, 2048)
    shapes = [u, u, w, bc, bc, (5120,), None, (5120,)]
    for at, two in (({}, True), ({0: (0, 0)}, False), ({1: (2, 0)}, False), ({1: (5, 0)}, False), ({0: (4, 64)}, False),
                    ({1: (7, 5120 * 4 - 4)}, False), ({1: (7, 5120 * 4)}, True)):
        got = launches("selective_scan", shapes, 2, at, return_last_state=1)
        assert (got == ["SelectiveScanFwdKernel"] * 2) == two and len(got) == 1 + two, (at, xp.last_launches())


@pytest.mark.parametrize("at,refused", [(7, False), (0, True), (3, True)])
def test_noalloc_decode_of_many_heads(at, refused):
    """A call of a few tokens needs none of the fixed array, so its heads are not
    limited by it; the chunked path, which an output over q or g takes, is."""
    k, state = (4096, 1, 16, 128), (4096, 16, 128, 128)
    ins = (_capi.XmTensor * 7)(*[xp._desc_from_shape(sh, (i + 1) << 34) for i, sh in enumerate([k] * 6 + [state])])
    a, err = xp._attrs("gated_deltanet2", scale=1.0), ctypes.create_string_buffer(512)
    st = xp.lib().xm_gated_deltanet2_forward_noalloc(ins, 7, ctypes.byref(a), (at + 1) << 34, None, err, len(err))
    assert (st == xp.XM_ERR_UNSUPPORTED) == refused, err.value
    assert xp.last_launches() == ([] if refused else ["Gdn2StepKernel<16,8>"])


def ss_launches(b, d, l, n, elem=1, var_c=True):
    row, bc, w = (b, d, l), (b, 1, n, l), (d, n)
    shapes = [row, row, w, bc, bc if var_c else w, (d,), None, (d,)]
    data = (0, 1, 3, 4) if var_c else (0, 1, 3)
    ins = (_capi.XmTensor * 8)(*[xp._desc_from_shape(sh, (i + 1) << 34, elem if i in data else 1) if sh is not None
                                 else xp._desc_from_tensor(None) for i, sh in enumerate(shapes)])
    a, err = xp._attrs("selective_scan"), ctypes.create_string_buffer(512)
    st = xp.lib().xm_selective_scan_forward(ins, 8, ctypes.byref(a), 9 << 34, None, None, err, len(err))
    names = [k.split("<")[0] for k in xp.last_launches()]
    return {("SelectiveScanFwdKernel",): "whole", ("SelectiveScanSegKernel",): "parallel",
            ("SelectiveScanFwdKernel",) * 2: "segments"}[tuple(names)]


@pytest.mark.parametrize("call,form", [   # where it was measured the cheapest by a quarter or more
    ((1, 256, 512, 16), "parallel"), ((1, 1024, 1999, 16), "parallel"), ((1, 5120, 1999, 16), "segments"),
    ((1, 4096, 1001, 16), "segments"), ((2, 4096, 1999, 16, _capi.XM_ELEM_BFLOAT16), "segments"),
    ((1, 2048, 1999, 64), "segments"), ((1, 4096, 512, 8), "parallel"), ((8, 5120, 2048, 16), "whole"),
    # guarded accesses make the whole pass and the segments slower than the sequence-parallel kernel
    ((8, 3403, 720, 3), "parallel"), ((2, 964, 5616, 8, _capi.XM_ELEM_FLOAT16), "parallel"),
    # a constant C
    ((7, 2971, 278, 1, _capi.XM_ELEM_FLOAT16, False), "parallel"), ((2, 12745, 1264, 1, _capi.XM_ELEM_BFLOAT16, False), "parallel"),
    ((1, 5120, 255, 16), "whole"),
], ids=str)
def test_ss_form(call, form):
    assert ss_launches(*call) == form, xp.last_launches()


def gdn2_launches(b, t, h, dk, dv):
    k, v, s = (b, t, h, dk), (b, t, h, dv), (b, h, dk, dv)
    return launches("gated_deltanet2", [k, k, v, k, k, v, s], 2, scale=1.0, output_final_state=1)


@pytest.mark.parametrize("call,step", [
    ((32, 16, 16, 128, 128), True), ((64, 16, 16, 64, 64), True), ((3072, 16, 1, 128, 64), True), ((1, 16, 4, 512, 8), True),
    ((3072, 4, 1, 16, 16), True), ((3072, 8, 1, 16, 16), False), ((192, 12, 16, 32, 16), False), ((1024, 6, 1, 512, 16), True),
    ((1024, 12, 1, 512, 16), False), ((2, 17, 2, 64, 64), False),
], ids=str)
def test_gdn2_step_or_chunked(call, step):
    """Without a GPU the chunked path ends at its scratch, before any launch."""
    assert gdn2_launches(*call) == (["Gdn2StepKernel"] if step else []), xp.last_launches()


@pytest.mark.parametrize("call,step", [
    ((2, 16, 128, 64, 128), True), ((1, 5, 104, 64, 16), True), ((1, 8, 104, 64, 16), False), ((298, 8, 1, 32, 32), True),
    ((298, 14, 1, 32, 32), False), ((61, 10, 6, 16, 64), False), ((61, 8, 6, 16, 64), True), ((720, 16, 1, 64, 32), True),
], ids=str)
def test_m3_step_or_chunked(call, step):
    b, t, h, p, n = call
    assert (m3_launches(b, t, h, p, n, n // 2) == STEP) == step, xp.last_launches()
