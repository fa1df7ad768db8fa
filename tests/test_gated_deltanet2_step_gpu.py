"""GatedDeltaNet2Fn for a few tokens (Gdn2StepKernel: the state through
registers in one launch) on the GPU vs the fp64 oracle: every key tiling at its
edges, value columns cut by a group of four or by a column block, both column
block widths, one to sixteen tokens (prepared four at a time), with and without
states, the L2 norm and an in-place state; 17 tokens and outputs over an input
that several column blocks read take the chunked path."""

import numpy as np
import pytest

import xmetai_onnx_plugins as xp
from oracle import cref
from parity import TOL_GDN2, TOL_GPU, check, to_dev
from xmetai_onnx_plugins import workloads as W

pytestmark = pytest.mark.gpu

KEYS = ("q", "k", "v", "g", "beta", "w", "initial_state")
S = W.GatedDeltaNet2Shape


def run(s, seed, **kw):
    inp = W.gated_deltanet2_inputs(s, seed=seed)
    o, f = xp.gated_deltanet2_fn(*(to_dev(inp[k]) for k in KEYS), scale=s.scale, use_qk_l2norm_in_kernel=s.l2norm,
                                 output_final_state=True, **kw)
    ref = cref.gated_deltanet2(*(inp[k] for k in KEYS), scale=s.scale, use_qk_l2norm=s.l2norm, dtype=np.float64,
                               return_state=True)
    return o.cpu().numpy(), f.cpu().numpy(), ref


def step_launched(columns):
    return xp.last_launches()[0].startswith(f"Gdn2StepKernel<{columns // 4},") and len(xp.last_launches()) == 1


@pytest.mark.parametrize("dk", [1, 5, 64, 65, 128, 129, 192, 200, 256, 300, 320, 384, 511, 512])
@pytest.mark.parametrize("tokens,dv", [(1, 64), (5, 33)])
def test_step_keys(dk, tokens, dv):
    o, f, ref = run(S(2, tokens, 3, dk, dv, per_key_gates=True), seed=dk)
    assert step_launched(32), xp.last_launches()
    check(f"gated_deltanet2_step/k{dk}_t{tokens}_v{dv}/o", o, ref[0], TOL_GDN2)
    check(f"gated_deltanet2_step/k{dk}_t{tokens}_v{dv}/s", f, ref[1], TOL_GDN2)


@pytest.mark.parametrize("dv", [1, 2, 3, 4, 31, 32, 33, 63, 65, 130])
@pytest.mark.parametrize("heads,columns", [(2, 32), (256, 64)])
def test_step_value_columns(dv, heads, columns):
    o, f, ref = run(S(2, 3, heads, 48, dv, per_key_gates=True), seed=dv)
    assert step_launched(columns), xp.last_launches()
    check(f"gated_deltanet2_step/v{dv}_{columns}/o", o, ref[0], TOL_GDN2)
    check(f"gated_deltanet2_step/v{dv}_{columns}/s", f, ref[1], TOL_GDN2)


@pytest.mark.parametrize("tokens", [1, 2, 4, 8, 9, 15, 16, 17])
@pytest.mark.parametrize("initial,l2norm", [(True, True), (False, True), (True, False)])
def test_step_tokens(tokens, initial, l2norm):
    s = S(2, tokens, 2, 128, 96, initial_state=initial, l2norm=l2norm)
    o, f, ref = run(s, seed=tokens)
    assert step_launched(32) == (tokens <= 16), xp.last_launches()
    # without the norm the state grows by |k|^2 a token, in any fp32 order (see tests/parity.py)
    inp = W.gated_deltanet2_inputs(s, seed=tokens)
    r32 = cref.gated_deltanet2(*(inp[k] for k in KEYS), scale=s.scale, use_qk_l2norm=l2norm, dtype=np.float32,
                               return_state=True)
    check(f"gated_deltanet2_step/t{tokens}_{initial}_{l2norm}/o", o, ref[0], TOL_GDN2, ref32=None if l2norm else r32[0])
    check(f"gated_deltanet2_step/t{tokens}_{initial}_{l2norm}/s", f, ref[1], TOL_GDN2, ref32=None if l2norm else r32[1])


def test_step_agrees_with_the_chunked_path(override):
    o, f, _ = run(S(3, 7, 4, 128, 128, per_key_gates=True), seed=3)
    assert step_launched(32)
    override("gdn2_path", 2)
    oc, fc, _ = run(S(3, 7, 4, 128, 128, per_key_gates=True), seed=3)
    assert any(k.startswith("Gdn2Chunk") for k in xp.last_launches()), xp.last_launches()
    check("gated_deltanet2_step/vs_chunked/o", o, oc, TOL_GPU)
    check("gated_deltanet2_step/vs_chunked/s", f, fc, TOL_GPU)


def call_states(dev, s, out_ptr, state_ptr):
    """xm_gated_deltanet2_forward_states on device tensors, outputs at the given addresses."""
    import ctypes
    import torch
    from xmetai_onnx_plugins import _capi
    arr = (_capi.XmTensor * 7)(*[xp._desc_from_tensor(x) for x in dev])
    attrs = xp._attrs("gated_deltanet2", scale=s.scale, output_final_state=1)
    err = ctypes.create_string_buffer(256)
    st = xp.lib().xm_gated_deltanet2_forward_states(arr, 7, ctypes.byref(attrs), out_ptr, state_ptr,
                                                    torch.cuda.current_stream().cuda_stream, None, err, len(err))
    assert st == xp.XM_OK, err.value
    torch.cuda.synchronize()


def test_step_state_in_place():
    """A decode loop may keep one state buffer: final_state over initial_state."""
    import torch
    s = S(2, 2, 4, 128, 64)
    inp = W.gated_deltanet2_inputs(s, seed=4)
    dev = [to_dev(inp[k]) for k in KEYS]
    o, f = xp.gated_deltanet2_fn(*dev, scale=s.scale, output_final_state=True)
    out = torch.empty_like(o)
    call_states(dev, s, out.data_ptr(), dev[6].data_ptr())
    assert torch.equal(out, o) and torch.equal(dev[6], f)


@pytest.mark.parametrize("tokens", [1, 6])
@pytest.mark.parametrize("key", KEYS[:6])
def test_outputs_over_an_input(key, tokens):
    """out over q, k, g or beta, which every column block of a head reads whole:
    the chunked path, which has read them before it writes; over v or w, which a
    block reads only in its own columns: still one launch."""
    import torch
    s = S(3, tokens, 8, 128, 128)
    inp = W.gated_deltanet2_inputs(s, seed=6)
    dev = [to_dev(inp[k]) for k in KEYS]
    o, f = xp.gated_deltanet2_fn(*dev, scale=s.scale, output_final_state=True)
    assert step_launched(32)
    state, at = torch.empty_like(f), KEYS.index(key)
    call_states(dev, s, dev[at].data_ptr(), state.data_ptr())
    assert step_launched(32) == (key in ("v", "w")), xp.last_launches()
    assert xp.last_launches()[-1].startswith(("Gdn2StepKernel<", "Gdn2ChunkRecurKernel<")), xp.last_launches()
    check(f"gated_deltanet2_step/over_{key}_t{tokens}/o", dev[at].cpu().numpy(), o.cpu().numpy(), TOL_GPU)
    check(f"gated_deltanet2_step/over_{key}_t{tokens}/s", state.cpu().numpy(), f.cpu().numpy(), TOL_GPU)


def test_outputs_over_a_part_of_an_input():
    """out one token row behind v; final_state over the end of g."""
    import torch
    s = S(1, 5, 4, 64, 64)
    inp = W.gated_deltanet2_inputs(s, seed=7)
    dev = [to_dev(inp[k]) for k in KEYS]
    o, f = xp.gated_deltanet2_fn(*dev, scale=s.scale, output_final_state=True)
    row = s.nheads * s.dv
    buf = torch.empty(o.numel() + row, device="cuda")
    v = buf[row:].view(o.shape)
    v.copy_(dev[2])
    state = torch.empty_like(f)
    call_states([*dev[:2], v, *dev[3:]], s, buf.data_ptr(), state.data_ptr())
    assert not step_launched(32), xp.last_launches()
    check("gated_deltanet2_step/behind_v/o", buf[:-row].view(o.shape).cpu().numpy(), o.cpu().numpy(), TOL_GPU)
    check("gated_deltanet2_step/behind_v/s", state.cpu().numpy(), f.cpu().numpy(), TOL_GPU)
    n = dev[3].numel()
    buf = torch.empty(n + f.numel() - 64, device="cuda")
    g = buf[:n].view(dev[3].shape)
    g.copy_(dev[3])
    call_states([*dev[:3], g, *dev[4:]], s, torch.empty_like(o).data_ptr(), buf[n - 64:].data_ptr())
    assert not step_launched(32), xp.last_launches()
    check("gated_deltanet2_step/over_g/s", buf[n - 64:].view(f.shape).cpu().numpy(), f.cpu().numpy(), TOL_GPU)
