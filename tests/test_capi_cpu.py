"""Host-side tests of the C ABI (no GPU): the library loads, exports every
function include/xmetai_recurrent.h declares, and its attribute checks and
shape validation reproduce the reference adapters' behaviour and messages
(selective_scan_fn_ort.cpp:50-117, mamba3_siso_fn_ort.cpp:43-227,
gated_deltanet2_fn_ort.cpp:46-219)."""

import ctypes
import os
import re
import subprocess

import pytest

import xmetai_onnx_plugins as xp
from xmetai_onnx_plugins import XmError, validate, check_attrs

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def header_functions(path):
    text = open(path).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(xm_[a-z0-9_]+)\s*\(", text)))


def test_header_lists_the_c_abi():
    fns = header_functions(os.path.join(ROOT, "include", "xmetai_recurrent.h"))
    assert sorted(fns) == sorted(xp.EXPORTED_SYMBOLS)


def test_library_exports_every_declared_symbol():
    lib = xp.lib()
    out = subprocess.run(["nm", "-D", "--defined-only", xp.LIB_PATH], capture_output=True, text=True, check=True).stdout
    exported = set(re.findall(r" T (\w+)$", out, flags=re.M))
    for name in header_functions(os.path.join(ROOT, "include", "xmetai_recurrent.h")):
        assert name in exported, name
        assert getattr(lib, name) is not None
    assert "gfx950" in xp.version()


def test_no_cpu_fallback_symbols():
    # The library is device code plus validation; it must not carry a host
    # implementation of the recurrences (those live only in oracle/).
    out = subprocess.run(["nm", "-DC", xp.LIB_PATH], capture_output=True, text=True, check=True).stdout
    assert "xmo_" not in out


# ---------------------------------------------------------------------------
# attributes (session-time checks, reference constructors)
# ---------------------------------------------------------------------------

def _attrs(op):
    t = xp._capi.OPS[op][0]()
    getattr(xp.lib(), f"xm_{op}_attrs_default")(ctypes.byref(t))
    return t


def test_attribute_defaults_match_reference():
    a = _attrs("selective_scan")
    assert (a.delta_softplus, a.return_last_state) == (0, 0)
    a = _attrs("mamba3_siso")
    assert (a.chunk_size, a.has_d, a.has_z, a.return_final_states, a.has_input_states, a.has_cu_seqlens) == (64, 1, 1, 0, 0, 0)
    a = _attrs("gated_deltanet2")
    assert a.scale == 1.0 and a.use_qk_l2norm_in_kernel == 1
    assert (a.output_final_state, a.use_gate_in_kernel, a.has_cu_seqlens, a.state_v_first) == (0, 0, 0, 0)


@pytest.mark.parametrize("op,kw,msg,status", [
    ("mamba3_siso", dict(chunk_size=0), "Mamba3SisoFn requires chunk_size > 0", xp.XM_ERR_INVALID_ARGUMENT),
    ("gated_deltanet2", dict(use_gate_in_kernel=1), "GatedDeltaNet2Fn v1 expects pre-applied gate tensors and does not support use_gate_in_kernel", xp.XM_ERR_UNSUPPORTED),
    ("gated_deltanet2", dict(state_v_first=1), "GatedDeltaNet2Fn v1 expects state layout (batch, head, key, value)", xp.XM_ERR_UNSUPPORTED),
    ("gated_deltanet2", dict(scale=0.0), "GatedDeltaNet2Fn requires a positive finite scale", xp.XM_ERR_INVALID_ARGUMENT),
    ("gated_deltanet2", dict(scale=-1.0), "GatedDeltaNet2Fn requires a positive finite scale", xp.XM_ERR_INVALID_ARGUMENT),
    ("gated_deltanet2", dict(scale=float("inf")), "GatedDeltaNet2Fn requires a positive finite scale", xp.XM_ERR_INVALID_ARGUMENT),
    ("gated_deltanet2", dict(scale=float("nan")), "GatedDeltaNet2Fn requires a positive finite scale", xp.XM_ERR_INVALID_ARGUMENT),
])
def test_attribute_rejections(op, kw, msg, status):
    with pytest.raises(XmError) as e:
        check_attrs(op, **kw)
    assert e.value.message == msg
    assert e.value.status == status


def test_attribute_check_order_matches_reference():
    # The GDN-2 constructor checks use_gate_in_kernel, cu_seqlens and the
    # state layout before the scale (gated_deltanet2_fn_ort.cpp:49-63).
    with pytest.raises(XmError, match="use_gate_in_kernel"):
        check_attrs("gated_deltanet2", use_gate_in_kernel=1, scale=-1.0)
    with pytest.raises(XmError, match="state layout"):
        check_attrs("gated_deltanet2", state_v_first=1, scale=float("nan"))


def test_state_attributes_are_accepted():
    # Widening: the reference rejects these; here they select the state
    # outputs of the *_forward_states entry points (and Mamba-3's state inputs).
    check_attrs("selective_scan", return_last_state=1, delta_softplus=1)
    check_attrs("gated_deltanet2", output_final_state=1, scale=0.5)
    check_attrs("mamba3_siso", return_final_states=1, has_input_states=1)
    check_attrs("mamba3_siso", has_cu_seqlens=1)
    check_attrs("gated_deltanet2", has_cu_seqlens=1)


def _forward_host_error(op, shapes, entry, state_ptrs=(None,), **attrs):
    """Calls a forward entry point on shape-only descriptors with a host-side
    error expected before any device work; returns (status, message)."""
    n = len(shapes)
    arr = (xp._capi.XmTensor * n)(*[xp._desc_from_shape(sh if sh is not None else (0,)) for sh in shapes])
    a = xp._attrs(op, **attrs)
    err = ctypes.create_string_buffer(512)
    fn = getattr(xp.lib(), f"xm_{op}_{entry}")
    out = ctypes.c_void_p(16)   # never dereferenced: every call below fails on the host first
    if entry == "forward":
        st = fn(arr, n, ctypes.byref(a), out, None, None, err, len(err))
    else:
        st = fn(arr, n, ctypes.byref(a), out, *state_ptrs, None, None, err, len(err))
    return st, err.value.decode()


def test_plain_forward_refuses_a_state_request():
    st, msg = _forward_host_error("selective_scan", ss_shapes(), "forward", return_last_state=1)
    assert st == xp.XM_ERR_INVALID_ARGUMENT and "xm_selective_scan_forward_states" in msg
    st, msg = _forward_host_error("gated_deltanet2", gdn_shapes(), "forward", output_final_state=1)
    assert st == xp.XM_ERR_INVALID_ARGUMENT and "xm_gated_deltanet2_forward_states" in msg
    st, msg = _forward_host_error("mamba3_siso", m3_shapes(), "forward", return_final_states=1, has_z=0)
    assert st == xp.XM_ERR_INVALID_ARGUMENT and "xm_mamba3_siso_forward_states" in msg


def test_states_entry_needs_a_state_buffer():
    st, msg = _forward_host_error("selective_scan", ss_shapes(), "forward_states", (None,), return_last_state=1)
    assert (st, msg) == (xp.XM_ERR_INVALID_ARGUMENT, "return_last_state=1 needs a last_state buffer")
    st, msg = _forward_host_error("gated_deltanet2", gdn_shapes(), "forward_states", (None,), output_final_state=1)
    assert (st, msg) == (xp.XM_ERR_INVALID_ARGUMENT, "output_final_state=1 needs a final_state buffer")
    some = (ctypes.c_void_p(16), ctypes.c_void_p(16), None, ctypes.c_void_p(16))   # one of the four missing
    st, msg = _forward_host_error("mamba3_siso", m3_shapes(), "forward_states", some, return_final_states=1, has_z=0)
    assert (st, msg) == (xp.XM_ERR_INVALID_ARGUMENT, "return_final_states=1 needs four state buffers")


def test_gdn2_scratch_follows_the_kernel_that_runs():
    """The planned scratch is the chunked path's by default and 0 when the
    gdn2_path override runs the sequential fused kernel (dk <= 512), which
    takes none; above 512 keys only the LDS-state path runs, with scratch."""
    import xmetai_onnx_plugins as xp
    def scratch(T, K, V):
        return validate("gated_deltanet2", gdn_shapes(T=T, K=K, V=V))[1]
    assert scratch(300, 128, 64) > 0
    assert scratch(3000, 512, 64) > 0
    with xp.kernel_override("gdn2_path", 1):
        assert scratch(300, 128, 64) == 0
        assert scratch(3000, 512, 64) == 0
        assert scratch(3000, 600, 64) > 0
    assert scratch(300, 128, 64) > 0


def test_states_entry_validates_shapes_first():
    bad = ss_shapes()
    bad[1] = (2, 8, 15)
    st, msg = _forward_host_error("selective_scan", bad, "forward_states", (None,), return_last_state=1)
    assert st == xp.XM_ERR_INVALID_ARGUMENT and "needs a last_state buffer" not in msg


# ---------------------------------------------------------------------------
# SelectiveScanFn shapes
# ---------------------------------------------------------------------------

def ss_shapes(B=2, D=8, L=16, N=4, G=None, bvar=True, cvar=True, has_d=True, has_z=True, has_bias=True):
    def bc(var):
        if not var:
            return (D, N)
        return (B, N, L) if G is None else (B, G, N, L)
    return [(B, D, L), (B, D, L), (D, N), bc(bvar), bc(cvar), (D,) if has_d else None,
            (B, D, L) if has_z else None, (D,) if has_bias else None]


@pytest.mark.parametrize("kw", [dict(), dict(G=2), dict(bvar=False), dict(cvar=False), dict(bvar=False, cvar=False),
                                dict(has_d=False, has_z=False, has_bias=False), dict(N=256), dict(N=1)])
def test_ss_valid_shapes(kw):
    shapes = ss_shapes(**kw)
    out, scratch = validate("selective_scan", shapes, delta_softplus=1)
    assert out == shapes[0]
    assert scratch == 0


@pytest.mark.parametrize("mutate,msg", [
    (lambda s: s.__setitem__(0, (2, 8)), "u must be 3-D"),
    (lambda s: s.__setitem__(1, (2, 8, 15)), "delta must have same shape as u"),
    (lambda s: s.__setitem__(2, (8, 4, 1)), "A must be 2-D"),
    (lambda s: s.__setitem__(3, (8,)), "B must have rank >= 2"),
    (lambda s: s.__setitem__(4, (4,)), "C must have rank >= 2"),
    (lambda s: s.__setitem__(2, (7, 4)), "A dimension mismatch with u"),
    (lambda s: (s.__setitem__(2, (8, 257)), s.__setitem__(3, (2, 257, 16)), s.__setitem__(4, (2, 257, 16))),
     "selective_scan supports d_state up to 256"),
    (lambda s: (s.__setitem__(3, (2, 3, 4, 16)), s.__setitem__(4, (2, 3, 4, 16))), "dim must be divisible by n_groups"),
])
def test_ss_reference_rejections(mutate, msg):
    shapes = ss_shapes()
    mutate(shapes)
    with pytest.raises(XmError) as e:
        validate("selective_scan", shapes)
    assert e.value.message == msg
    assert e.value.status == xp.XM_ERR_INVALID_ARGUMENT


@pytest.mark.parametrize("idx,shape,msg", [
    (3, (2, 4, 15), "B must have shape (batch, n_groups, dstate, seqlen) when variable"),
    (3, (3, 4, 16), "B must have shape (batch, n_groups, dstate, seqlen) when variable"),
    (4, (2, 5, 16), "C must have shape (batch, n_groups, dstate, seqlen) when variable"),
    (5, (7,), "D must have shape (dim,)"),
    (6, (2, 8, 15), "z must have same shape as u"),
    (7, (9,), "delta_bias must have shape (dim,)"),
])
def test_ss_extent_checks_beyond_reference(idx, shape, msg):
    # The reference does not check these extents and reads out of bounds on them.
    shapes = ss_shapes()
    shapes[idx] = shape
    with pytest.raises(XmError) as e:
        validate("selective_scan", shapes)
    assert e.value.message == msg


@pytest.mark.parametrize("kw", [dict(), dict(bvar=False, cvar=False), dict(has_d=False)])
def test_ss_dstate_zero_is_accepted_like_reference(kw):
    # The reference only caps d_state at 256 (selective_scan_fn_ort.cpp:99-105);
    # with d_state = 0 its state loop is empty and y = D * u.
    out, scratch = validate("selective_scan", ss_shapes(N=0, **kw))
    assert out == (2, 8, 16) and scratch == 0


def test_kernel_overrides_roundtrip():
    from xmetai_onnx_plugins import _capi
    for name, values in _capi.KERNEL_OVERRIDES.items():
        assert xp.get_kernel_override(name) == 0
        for v in values:
            with xp.kernel_override(name, v):
                assert xp.get_kernel_override(name) == v
        assert xp.get_kernel_override(name) == 0
    assert xp.get_kernel_override("no_such_switch") == -1
    with pytest.raises(XmError) as e:
        xp.set_kernel_override("no_such_switch", 1)
    assert e.value.status == xp.XM_ERR_INVALID_ARGUMENT
    with pytest.raises(XmError):
        xp.set_kernel_override("ss_lpc", 3)
    assert xp.get_kernel_override("ss_lpc") == 0


def test_ss_empty_sequence_is_a_no_op():
    out, _ = validate("selective_scan", ss_shapes(L=0))
    assert out == (2, 8, 0)


SS_TYPES_MSG = ("SelectiveScanFn: u, delta, z and variable B/C must share one element type; "
                "constant B/C are float32")


@pytest.mark.parametrize("half", [10, 16])   # FLOAT16, BFLOAT16
def test_ss_16bit_data_types(half):
    # Widening: u, delta, z and variable B/C in one 16-bit type (the reference's
    # half / bfloat16 kernels); A, D, delta_bias and constant B/C stay float32.
    data = [half, half, 1, half, half, 1, half, 1]
    assert validate("selective_scan", ss_shapes(), data)[0] == (2, 8, 16)
    const_b = [half, half, 1, 1, half, 1, half, 1]
    assert validate("selective_scan", ss_shapes(bvar=False), const_b)[0] == (2, 8, 16)
    for types, shapes, msg in (
            ([1, half, 1, 1, 1, 1, 1, 1], ss_shapes(), SS_TYPES_MSG),             # mixed data types
            ([half, half, 1, half, 1, 1, half, 1], ss_shapes(), SS_TYPES_MSG),    # variable C in fp32
            ([half, half, 1, half, half, 1, 1, 1], ss_shapes(), SS_TYPES_MSG),    # z in fp32
            ([half, half, 1, half, half, 1, half, 1], ss_shapes(bvar=False), SS_TYPES_MSG),   # 16-bit constant B
            ([half, half, half, half, half, 1, half, 1], ss_shapes(), "TensorView expects float32 tensors"),   # A
            ([half, half, 1, half, half, half, half, 1], ss_shapes(), "TensorView expects float32 tensors"),   # D
            ([7, 7, 1, 7, 7, 1, 7, 1], ss_shapes(), "TensorView expects float32 tensors")):  # int64 data
        with pytest.raises(XmError) as e:
            validate("selective_scan", shapes, types)
        assert e.value.message == msg


def test_wrong_input_count():
    with pytest.raises(TypeError):
        validate("selective_scan", ss_shapes()[:7])


class _LooksLikeATensor:
    """Not a tensor, but with what the descriptors are made from."""
    shape = (2, 8, 16)
    is_cuda = True
    dtype = None

    def data_ptr(self):
        return 16

    def numel(self):
        return 256

    def is_contiguous(self):
        return True


def test_front_end_refuses_what_is_no_device_tensor():
    import torch
    import xmetai_onnx_plugins as xp
    t = torch.zeros(2, 8, 16)
    with pytest.raises(TypeError, match="inputs must be torch tensors or None"):
        xp.selective_scan_fn(_LooksLikeATensor(), t, t, t, t)
    with pytest.raises(TypeError, match="inputs must be torch tensors or None"):
        xp.selective_scan_fn(t.numpy(), t, t, t, t)
    for x in (t, t.to_sparse(), t.transpose(1, 2)):   # a sparse tensor has no address to ask for
        with pytest.raises(XmError, match="inputs must be device tensors"):
            xp.selective_scan_fn(x, t, t, t, t)


# ---------------------------------------------------------------------------
# GatedDeltaNet2Fn shapes
# ---------------------------------------------------------------------------

def gdn_shapes(B=2, T=5, H=3, K=16, V=8, s0=True):
    qk = (B, T, H, K)
    vv = (B, T, H, V)
    return [qk, qk, vv, qk, qk, vv, (B, H, K, V) if s0 else None]


def test_gdn2_valid_and_scratch():
    out, scratch = validate("gated_deltanet2", gdn_shapes(), scale=0.25)
    assert out == (2, 5, 3, 8)
    a256 = lambda n: (n + 255) // 256 * 256

    # headdim_k <= 512 (chunked path): per (b,h) and 16-token chunk of a window
    # of up to 128 chunks, E, R, Ut tiles (256 floats per 16 keys each), M T
    # (256), and per recurrence wave ceil((8 + 4 kpw) / 16) scalar vectors of
    # 64 floats (q and k multipliers, G_15);
    # keys padded to 16 * kpw * ks (kpw = 2 and ks = ceil(tiles / 2) up to 128
    # keys; 3 tiles x 4 waves for 129-192 keys; 5 tiles x 4 waves for 257-320
    # keys; for 321-384 keys 3 tiles x 8 waves when the launch has fewer than
    # 128 column-tile workgroups, else 6 tiles x 4 waves; else kpw = 4 and
    # ks = ceil(tiles / 4));
    # plus the state carried between windows when there is more than one
    def chunk_scratch(B, T, H, K, V):
        kq = -(-K // 16)
        groups = B * H * -(-V // 16)
        if 8 < kq <= 12:
            kpw, ks = 3, 4
        elif 16 < kq <= 20:
            kpw, ks = 5, 4
        elif 20 < kq <= 24:
            kpw, ks = (3, 8) if groups < 128 else (6, 4)
        elif kq > 8:
            kpw, ks = 4, -(-kq // 4)
        else:
            kpw = 2 if kq >= 2 else 1
            ks = -(-kq // kpw)
        kq = kpw * ks
        block = 3 * kq * 256 + 256 + ks * (-(-(8 + 4 * kpw) // 16)) * 64
        nch = -(-T // 16)
        rows, vt, kt = B * H, -(-V // 16), -(-K // 16)
        # sequence split, 64+ chunks: rows (vt + kt) <= 160 column tiles,
        # max(2, min(ceil(chunks / 64), 1 + ceil(1536 / (rows (vt + kt))))) segments;
        # above 160, two segments when rows vt <= 64 and rows vt + rows (vt + kt)
        # <= 256, or (two-tile split: a two-tile kernel for the key tiling, up to
        # 256 keys) when rows (vt + ceil(vt / 2) + ceil(kt / 2)) <= 256 CUs; every
        # chunk's blocks, Psi [B,T,H,KP], Phi [nseg][rows][K][KP] (KP = 16 kt), S0
        # and the start states [nseg][rows][K][V]; at most 2 GiB
        wide = rows * (vt + kt) > 160
        two_tile = (kpw, ks) in ((2, 2), (2, 3), (2, 4), (3, 4), (4, 4))
        if (nch >= 64 and nch * block * 4 < (1 << 31)
                and (not wide or (rows * vt <= 64 and rows * vt + rows * (vt + kt) <= 256)
                     or (two_tile and rows * (vt + -(-vt // 2) + -(-kt // 2)) <= 256))):
            nseg = 2 if wide else max(2, min(-(-nch // 64), 1 + -(-1536 // (rows * (vt + kt)))))
            sc = -(-nch // nseg)
            nseg = -(-nch // sc)
            if nseg >= 2:
                total = (a256(rows * nch * block * 4) + a256(B * T * H * kt * 16 * 4)
                         + a256(nseg * rows * K * kt * 16 * 4) + 2 * a256(nseg * rows * K * V * 4))
                if total <= 2 << 30:
                    return total
        # windows of 128 chunks, or of up to 128 MiB of blocks, balanced in length
        per_block = B * H * block * 4
        win = min(nch, 128)
        fit = min((128 << 20) // per_block, nch)
        if fit > win:
            win = -(-nch // -(-nch // fit))
        return a256(per_block * win) + (a256(B * H * K * V * 4) if win < nch else 0)
    assert scratch == chunk_scratch(2, 5, 3, 16, 8)
    for T, K, V in ((100, 128, 64), (3000, 128, 128), (17, 100, 7), (2049, 256, 16), (2048, 33, 40),
                    (3000, 512, 64), (40, 300, 16), (40, 352, 16), (40, 352, 352), (33, 385, 8), (50, 129, 8), (50, 150, 8), (50, 192, 8), (50, 80, 8), (50, 96, 8), (50, 48, 8),
                    (2048, 320, 64), (2048, 384, 64), (2048, 512, 64),
                    (2048, 256, 256), (2048, 200, 240), (1024, 256, 256), (1008, 256, 256),
                    (2048, 320, 256), (2048, 128, 640)):
        assert validate("gated_deltanet2", gdn_shapes(T=T, K=K, V=V))[1] == chunk_scratch(2, T, 3, K, V), (T, K, V)
    # packed sequences (headdim_k <= 512) take the fused kernel: no scratch
    # headdim_k > 512: prepared chunk of B*H*min(T,1024) rows (4 vectors x K padded
    # to 64) + one q.k float per row, plus the carried state when T > 1024
    _, s_short = validate("gated_deltanet2", gdn_shapes(T=100, K=600, V=64))
    assert s_short == a256(2 * 3 * 100 * 4 * 640 * 4) + a256(2 * 3 * 100 * 4)
    _, s_long = validate("gated_deltanet2", gdn_shapes(T=3000, K=600, V=64))
    rows = 2 * 3 * 1024
    assert s_long == a256(rows * 4 * 640 * 4) + a256(rows * 4) + 2 * 3 * 600 * 64 * 4


@pytest.mark.parametrize("idx,shape,msg", [
    (0, (2, 5, 3), "q must have rank 4"),
    (1, (2, 5, 3, 8), "q shape must match k"),
    (3, (2, 5, 3, 8), "q shape must match g"),
    (4, (2, 5, 3, 8), "q shape must match beta"),
    (2, (2, 4, 3, 8), "v batch/seqlen/head dimensions must match q"),
    (5, (2, 5, 3, 7), "v shape must match w"),
    (6, (2, 3, 16), "initial_state must have rank 4"),
    (6, (2, 3, 16, 9), "initial_state must have shape (batch, head, headdim_k, headdim_v)"),
])
def test_gdn2_reference_rejections(idx, shape, msg):
    shapes = gdn_shapes()
    shapes[idx] = shape
    with pytest.raises(XmError) as e:
        validate("gated_deltanet2", shapes)
    assert e.value.message == msg


def test_gdn2_zero_dims_rejected_like_reference():
    with pytest.raises(XmError, match="seqlen dimension is out of range"):
        validate("gated_deltanet2", gdn_shapes(T=0))


I64 = xp._capi.XM_ELEM_INT64


def packed_gdn(N=3, T=20, H=3, K=16, V=8, s0=True, cu=None):
    shapes = gdn_shapes(B=1, T=T, H=H, K=K, V=V, s0=False)
    shapes[6] = (N, H, K, V) if s0 else None
    return shapes + [cu or (N + 1,)], [1] * 7 + [I64]


def packed_chunk_scratch(N, T, H, K, V):
    """Scratch of the chunked path for N packed sequences along T tokens.  A
    window holds chunks [c0, c0 + win) of every sequence (win = min(ceil(T/16),
    128), or every chunk when that costs at most twice the blocks or 512 MiB);
    per head its blocks are at most min(win * N, ceil(T/16) + N), of
    3*kq*256 + 16*kq + 288 floats each (kq = key tiles, padded to the
    recurrence's key split).  Plus the carried state [N,H,K,V] when a sequence
    can span windows, and the per-window block offsets [windows][N+1] ints;
    each region 256-byte aligned."""
    a256 = lambda x: -(-x // 256) * 256
    kq = -(-K // 16)   # (the key layouts of 16, 64, 128, 256 and 512 keys)
    kpw = 4 if kq > 8 else (1 if kq < 2 else 2)
    ks = -(-kq // kpw)
    kq = kpw * ks
    nch = -(-T // 16)
    per = H * (3 * kq * 256 + 256 + ks * (-(-(8 + 4 * kpw) // 16)) * 64) * 4
    win = min(nch, 128)
    blocks = a256(per * min(win * N, nch + N))
    if win < nch and a256(per * (nch + N)) <= max(2 * blocks, 512 << 20):
        win = nch   # one window over every chunk: no empty windows to step through
        blocks = a256(per * (nch + N))
    carry = a256(N * H * K * V * 4) if win < nch else 0
    return blocks + carry + a256(-(-nch // win) * (N + 1) * 4)


def test_gdn2_packed_sequences_valid_scratch():
    # Widening: cu_seqlens (input 7, int64 [N+1]) packs N sequences; the
    # chunked path takes them at any headdim_k up to 512, with global-chunk
    # windows and the chunk offsets in scratch.
    for K in (16, 128, 256, 512):
        shapes, types = packed_gdn(K=K)
        assert validate("gated_deltanet2", shapes, types, has_cu_seqlens=1) == \
            ((1, 20, 3, 8), packed_chunk_scratch(3, 20, 3, K, 8))
    # 4000 tokens in 5 sequences: one window over every chunk
    shapes, types = packed_gdn(N=5, T=4000, K=64)
    assert validate("gated_deltanet2", shapes, types, has_cu_seqlens=1)[1] == packed_chunk_scratch(5, 4000, 3, 64, 8)
    # one 2^20-token sequence at 16 x 256 x 256: windows of 128 chunks, the state carried
    shapes, types = packed_gdn(N=1, T=1 << 20, H=16, K=256, V=256)
    assert validate("gated_deltanet2", shapes, types, has_cu_seqlens=1)[1] == \
        packed_chunk_scratch(1, 1 << 20, 16, 256, 256)
    shapes, types = packed_gdn(s0=False)
    assert validate("gated_deltanet2", shapes, types, has_cu_seqlens=1)[0] == (1, 20, 3, 8)


@pytest.mark.parametrize("mutate,msg", [
    (lambda s, t: s.__setitem__(0, (2, 20, 3, 16)),
     "GatedDeltaNet2Fn with cu_seqlens requires batch 1 (sequences packed along seqlen)"),
    (lambda s, t: s.__setitem__(6, (1, 3, 16, 8)), "initial_state must have shape (sequences, head, headdim_k, headdim_v)"),
    (lambda s, t: t.__setitem__(7, 1), "cu_seqlens must be an int64 tensor"),
    (lambda s, t: s.__setitem__(7, (2, 2)), "cu_seqlens must have rank 1"),
    (lambda s, t: s.__setitem__(7, (1,)), "cu_seqlens must hold at least two offsets"),
])
def test_gdn2_packed_sequences_rejections(mutate, msg):
    shapes, types = packed_gdn()
    mutate(shapes, types)
    if shapes[0][0] == 2:   # the other q-shaped inputs follow q
        shapes[1:6] = [(2,) + tuple(x[1:]) for x in shapes[1:6]]
    with pytest.raises(XmError) as e:
        validate("gated_deltanet2", shapes, types, has_cu_seqlens=1)
    assert e.value.message == msg


def test_gdn2_packed_sequences_limits():
    shapes, types = packed_gdn(K=600)
    with pytest.raises(XmError, match="with cu_seqlens supports headdim_k up to 512"):
        validate("gated_deltanet2", shapes, types, has_cu_seqlens=1)
    with pytest.raises(XmError, match="expects 8 inputs, got 7"):
        validate("gated_deltanet2", gdn_shapes(B=1), has_cu_seqlens=1)


def test_gdn2_absent_initial_state():
    out, _ = validate("gated_deltanet2", gdn_shapes(s0=False))
    assert out == (2, 5, 3, 8)


# ---------------------------------------------------------------------------
# Mamba3SisoFn shapes
# ---------------------------------------------------------------------------

def m3_shapes(B=2, T=7, H=4, Hq=2, P=8, N=16, A=8, has_d=True, has_z=False):
    return [(B, T, Hq, N), (B, T, Hq, N), (B, T, H, P), (B, H, T), (B, H, T), (B, H, T), (H, N), (H, N),
            (B, T, H, A), (H,) if has_d else None, (B, T, H, P) if has_z else None]


def m3_state_shapes(B=2, H=4, P=8, N=16, A=8):
    return [(B, H, P, N), (B, H, A), (B, H, N), (B, H, P)]


def test_m3_input_states_take_inputs_11_to_14():
    # Widening: has_input_states=1 adds the four states as inputs 11-14.
    out, scratch = validate("mamba3_siso", m3_shapes() + m3_state_shapes(), has_input_states=1, has_z=0)
    assert out == (2, 7, 4, 8) and scratch == 0
    with pytest.raises(XmError, match="expects 15 inputs, got 11"):
        validate("mamba3_siso", m3_shapes(), has_input_states=1, has_z=0)
    with pytest.raises(XmError, match="expects 11 inputs, got 15"):
        validate("mamba3_siso", m3_shapes() + m3_state_shapes(), has_z=0)


@pytest.mark.parametrize("i,shape,msg", [
    (0, (2, 4, 16, 8), "ssm_state must have shape (batch, nheads, headdim_v, headdim_qk)"),
    (0, (2, 4, 8), "ssm_state must have rank 4"),
    (1, (2, 4, 7), "angle_state must have shape (batch, nheads, headdim_angles)"),
    (2, (2, 2, 16), "k_state must have shape (batch, nheads, headdim_qk)"),
    (3, (2, 4, 16), "v_state must have shape (batch, nheads, headdim_v)"),
    (3, None, "v_state must have rank 3"),
])
def test_m3_input_state_shapes(i, shape, msg):
    st = m3_state_shapes()
    st[i] = shape
    with pytest.raises(XmError) as e:
        validate("mamba3_siso", m3_shapes() + st, has_input_states=1, has_z=0)
    assert e.value.message == msg


def test_m3_packed_sequences():
    # Widening: cu_seqlens is input 15 (16 inputs; the state slots 11-14 stay
    # empty without has_input_states).
    base = m3_shapes(B=1, T=30)
    types = [1] * 15 + [I64]
    out, scratch = validate("mamba3_siso", base + [None] * 4 + [(4,)], types, has_cu_seqlens=1, has_z=0)
    assert out == (1, 30, 4, 8) and scratch == 0
    st = m3_state_shapes(B=3)
    assert validate("mamba3_siso", base + st + [(4,)], types, has_cu_seqlens=1, has_input_states=1, has_z=0)[0] == \
        (1, 30, 4, 8)
    with pytest.raises(XmError, match="state inputs need has_input_states=1"):
        validate("mamba3_siso", base + st + [(4,)], types, has_cu_seqlens=1, has_z=0)
    with pytest.raises(XmError, match="ssm_state must have shape"):
        validate("mamba3_siso", base + m3_state_shapes(B=1) + [(4,)], types, has_cu_seqlens=1, has_input_states=1,
                 has_z=0)
    with pytest.raises(XmError, match="requires batch 1"):
        validate("mamba3_siso", m3_shapes(B=2) + [None] * 4 + [(4,)], types, has_cu_seqlens=1, has_z=0)
    with pytest.raises(XmError, match="cu_seqlens must be an int64 tensor"):
        validate("mamba3_siso", base + [None] * 4 + [(4,)], [1] * 16, has_cu_seqlens=1, has_z=0)


def test_m3_valid():
    out, scratch = validate("mamba3_siso", m3_shapes(), has_d=1, has_z=0)
    assert out == (2, 7, 4, 8) and scratch == 0
    # any even headdim_qk: above 512 keys one launch per 512-key block (the
    # reference's shared-memory budget allows N = 576 at P = 64, ~2000 at P = 16)
    assert validate("mamba3_siso", m3_shapes(P=64, N=512, A=256), has_d=1, has_z=0)[0] == (2, 7, 4, 64)
    assert validate("mamba3_siso", m3_shapes(P=64, N=514, A=256), has_d=1, has_z=0)[0] == (2, 7, 4, 64)
    assert validate("mamba3_siso", m3_shapes(P=16, N=2048, A=100), has_d=1, has_z=0)[0] == (2, 7, 4, 16)
    out, _ = validate("mamba3_siso", m3_shapes(has_z=True), has_d=1, has_z=1)
    assert out == (2, 7, 4, 8)


@pytest.mark.parametrize("mutate,attrs,msg", [
    (lambda s: s.__setitem__(3, (2, 4)), {}, "ADT must have rank 3"),
    (lambda s: s.__setitem__(1, (2, 7, 2, 14)), {}, "Q shape must match K"),
    (lambda s: s.__setitem__(4, (2, 4, 6)), {}, "ADT shape must match DT"),
    (lambda s: s.__setitem__(2, (2, 6, 4, 8)), {}, "V batch/seqlen must match Q"),
    (lambda s: s.__setitem__(6, (4, 14)), {}, "Q_bias must have shape (nheads, headdim_qk)"),
    (lambda s: s.__setitem__(8, (2, 7, 3, 8)), {}, "Angles must have shape (batch, seqlen, nheads, headdim_angles)"),
    (lambda s: s.__setitem__(8, (2, 7, 4, 9)), {}, "Mamba3SisoFn requires 0 < headdim_angles <= headdim_qk / 2"),
    (lambda s: s.__setitem__(9, None), {}, "Mamba3SisoFn has_d attribute does not match D input"),
    (lambda s: s.__setitem__(10, (2, 7, 4, 8)), {}, "Mamba3SisoFn has_z attribute does not match Z input"),
    (lambda s: s.__setitem__(9, (3,)), {}, "D must have shape (nheads,)"),
])
def test_m3_reference_rejections(mutate, attrs, msg):
    shapes = m3_shapes()
    mutate(shapes)
    with pytest.raises(XmError) as e:
        validate("mamba3_siso", shapes, has_d=1, has_z=0, **attrs)
    assert e.value.message == msg


def test_m3_head_divisibility_and_odd_dim():
    with pytest.raises(XmError, match="nheads divisible by nheads_qk"):
        validate("mamba3_siso", m3_shapes(H=3, Hq=2), has_d=1, has_z=0)
    shapes = m3_shapes(N=15, A=4)
    with pytest.raises(XmError, match="positive even headdim_qk"):
        validate("mamba3_siso", shapes, has_d=1, has_z=0)


# ---------------------------------------------------------------------------
# ONNX Runtime layer (compiled only where ORT headers exist; its contract with
# the reference is checked on the sources here)
# ---------------------------------------------------------------------------

ORT_DIR = os.path.join(ROOT, "xmetai-onnx-plugins_amd", "csrc", "ort")


def _src(name):
    with open(os.path.join(ORT_DIR, name)) as f:
        return f.read()


def test_ort_header_declares_register_custom_ops():
    with open(os.path.join(ROOT, "include", "xmetai_onnx_plugins_ort.h")) as f:
        h = f.read()
    assert "OrtStatus *ORT_API_CALL RegisterCustomOps(OrtSessionOptions *options, const OrtApiBase *api_base);" in h


def test_ort_registration_domain_and_order():
    # reference register_op.cpp:20-40: domain xmetai_plugins, ops in this order
    reg = _src("register_op.cpp")
    assert 'extern "C" OrtStatus *ORT_API_CALL RegisterCustomOps' in reg
    assert 'kDomain = "xmetai_plugins"' in _src("ort_glue.h")
    order = ["XmAddSelectiveScanFnOp", "XmAddMamba3SisoFnOp", "XmAddGatedDeltaNet2FnOp", "XmAddSoftmaxCpuOp"]
    line = [l for l in reg.splitlines() if "const AddFn adds[]" in l][0]
    assert [line.index(n) for n in order] == sorted(line.index(n) for n in order)


def test_ort_descriptors_match_reference_contract():
    ops = _src("ops_ort.cpp")
    # output 1 (optional) is the state after the last token where the op has one
    # (Mamba-3: inputs 11-14 the input states, 15 cu_seqlens; GDN-2: 7 cu_seqlens; all optional)
    for name, n_in, n_out, n_req in (("SelectiveScanFn", 8, 2, 8), ("Mamba3SisoFn", 16, 5, 11),
                                     ("GatedDeltaNet2Fn", 8, 2, 7)):
        block = ops[ops.index(f'return "{name}";') - 400:ops.index(f'return "{name}";') + 1000]
        assert f"GetInputTypeCount() const {{ return {n_in}; }}" in block
        assert f"GetOutputTypeCount() const {{ return {n_out}; }}" in block
        assert "return i == 0 ? INPUT_OUTPUT_REQUIRED : INPUT_OUTPUT_OPTIONAL;" in block
        if n_req < n_in:
            assert f"return i < {n_req} ? INPUT_OUTPUT_REQUIRED : INPUT_OUTPUT_OPTIONAL;" in block
            assert f"return i == {n_in - 1} ? ONNX_TENSOR_ELEMENT_DATA_TYPE_INT64" in block
        else:
            assert "GetInputCharacteristic" not in block
        assert "GetExecutionProviderType() const { return XM_ORT_GPU_EP; }" in block
    for attr in ("delta_softplus", "return_last_state", "chunk_size", "has_d", "has_z", "return_final_states",
                 "has_input_states", "has_cu_seqlens", "scale", "use_qk_l2norm_in_kernel", "output_final_state",
                 "use_gate_in_kernel", "state_v_first"):
        assert f'"{attr}"' in ops
    # widening: float16 / bfloat16 SelectiveScanFn descriptors (data inputs 0, 1, 3, 4, 6 and y
    # 16-bit; A, D, delta_bias and the state float), added right after the float one
    assert "return (i <= 1 || i == 3 || i == 4 || i == 6) ? DT : ONNX_TENSOR_ELEMENT_DATA_TYPE_FLOAT;" in ops
    assert "return i == 0 ? DT : ONNX_TENSOR_ELEMENT_DATA_TYPE_FLOAT;" in ops
    add = ops[ops.index("OrtStatus *XmAddSelectiveScanFnOp"):]
    add = add[:add.index("\n}\n")]
    assert [add.index(g) for g in ("&g_selective_scan_op)", "&g_selective_scan_op_f16)",
                                   "&g_selective_scan_op_bf16)")] == sorted(
        add.index(g) for g in ("&g_selective_scan_op)", "&g_selective_scan_op_f16)", "&g_selective_scan_op_bf16)"))
    assert "SelectiveScanOpT<ONNX_TENSOR_ELEMENT_DATA_TYPE_FLOAT16> g_selective_scan_op_f16;" in ops
    assert "SelectiveScanOpT<ONNX_TENSOR_ELEMENT_DATA_TYPE_BFLOAT16> g_selective_scan_op_bf16;" in ops
    sm = _src("softmax_cpu_ort.cpp")
    assert 'return "SoftmaxCPU";' in sm and '"CPUExecutionProvider"' in sm and '"axis", -1' in sm
    assert '#define XM_ORT_GPU_EP "ROCMExecutionProvider"' in _src("ort_glue.h")


@pytest.mark.skipif(not os.path.exists(os.path.join(os.environ.get("ORT_INCLUDE_DIR", "/nonexistent"),
                                                    "onnxruntime_c_api.h")),
                    reason="ONNX Runtime headers are not installed (set ORT_INCLUDE_DIR)")
def test_ort_library_builds_and_exports_register_custom_ops():
    import ctypes
    import importlib.util
    spec = importlib.util.spec_from_file_location("xm_build", os.path.join(ROOT, "xmetai-onnx-plugins_amd", "build.py"))
    mod = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(mod)
    mod.build(ort_include=os.environ["ORT_INCLUDE_DIR"])
    assert hasattr(ctypes.CDLL(mod.ORT_LIB), "RegisterCustomOps")
