"""Packed sequences on the XCD-spread workgroup order (a sequence's heads over
all XCDs): unit counts that are no multiple of the 8 XCDs, several workgroups per
unit, more sequences than chunk slots, empty sequences, and token rows that no
sequence covers, against the same sequences run one by one."""

import numpy as np
import pytest

import xmetai_onnx_plugins as xp
from parity import TOL_GPU, check, to_dev
from xmetai_onnx_plugins import workloads as W

pytestmark = pytest.mark.gpu

OFFSETS = {
    "even": [0, 40, 80, 120],
    "one_long": [0, 3, 5, 150, 157],
    "empty_and_gaps": [4, 4, 60, 60, 61, 150],
    "one_token_each": list(range(0, 41)),
}


def single_runs(call, offsets, total, like):
    """Each sequence by itself; zeros where none covers a row."""
    out = np.zeros(like, np.float32)
    for lo, hi in zip(offsets, offsets[1:]):
        if hi > lo:
            out[:, lo:hi] = call(lo, hi)
    return out


@pytest.mark.parametrize("heads,dv", [(1, 16), (3, 64), (5, 200), (8, 40)])
@pytest.mark.parametrize("name", sorted(OFFSETS))
def test_gdn2_spread(name, heads, dv):
    off, total = OFFSETS[name], 160
    s = W.GatedDeltaNet2Shape(1, total, heads, 64, dv, initial_state=False, per_key_gates=True)
    inp = W.gated_deltanet2_inputs(s, seed=51)
    dev = [to_dev(inp[k]) for k in ("q", "k", "v", "g", "beta", "w")]
    got = xp.gated_deltanet2_fn(*dev, scale=s.scale, cu_seqlens=to_dev(np.asarray(off, np.int64))).cpu().numpy()
    want = single_runs(lambda lo, hi: xp.gated_deltanet2_fn(*(x[:, lo:hi].contiguous() for x in dev),
                                                            scale=s.scale).cpu().numpy(), off, total, got.shape)
    check(f"packed_spread/gdn2_{name}_h{heads}_v{dv}", got, want, TOL_GPU)


@pytest.mark.parametrize("heads,p", [(1, 16), (3, 64), (5, 100), (8, 32)])
@pytest.mark.parametrize("has_z", [True, False])
@pytest.mark.parametrize("name", sorted(OFFSETS))
def test_m3_spread(name, heads, p, has_z):
    off, total = OFFSETS[name], 160
    s = W.Mamba3SisoShape(1, total, heads, p, 64, has_z=has_z)
    inp = W.mamba3_siso_inputs(s, seed=52)
    keys = ("Q", "K", "V", "ADT", "DT", "Trap", "Q_bias", "K_bias", "Angles", "D", "Z")
    dev = {k: to_dev(inp[k]) for k in keys}

    def part(k, lo, hi):
        x = dev[k]
        if x is None or k in ("Q_bias", "K_bias", "D"):
            return x
        return (x[:, :, lo:hi] if k in ("ADT", "DT", "Trap") else x[:, lo:hi]).contiguous()
    got = xp.mamba3_siso_fn(*dev.values(), cu_seqlens=to_dev(np.asarray(off, np.int64))).cpu().numpy()
    want = single_runs(lambda lo, hi: xp.mamba3_siso_fn(*(part(k, lo, hi) for k in keys)).cpu().numpy(), off, total,
                       got.shape)
    check(f"packed_spread/m3_{name}_h{heads}_p{p}_{has_z}", got, want, TOL_GPU)


@pytest.mark.parametrize("dk,dv", [(64, 40), (128, 128), (128, 65), (192, 48), (256, 80)])
@pytest.mark.parametrize("offsets", [[0, 1500, 1540, 1600], [k * 100 for k in range(17)]], ids=["one_long", "even"])
def test_gdn2_tiles_by_length_equal_both_layouts_bitwise(dk, dv, offsets, override):
    """The packed recurrence picks one or two column tiles per workgroup from the
    lengths; either choice gives the bits of the fixed layouts."""
    s = W.GatedDeltaNet2Shape(1, 1600, 32, dk, dv, initial_state=False)
    inp = W.gated_deltanet2_inputs(s, seed=53)
    dev = [to_dev(inp[k]) for k in ("q", "k", "v", "g", "beta", "w")]
    cu = to_dev(np.asarray(offsets, np.int64))
    got = xp.gated_deltanet2_fn(*dev, scale=s.scale, cu_seqlens=cu)
    assert any(k.startswith("Gdn2ChunkRecurKernel<") and k.endswith(",0,1>") for k in xp.last_launches()), xp.last_launches()
    for ct in (1, 2):
        override("gdn2_ct", ct)
        fixed = xp.gated_deltanet2_fn(*dev, scale=s.scale, cu_seqlens=cu)
        assert np.array_equal(got.cpu().numpy(), fixed.cpu().numpy())


def many_lengths(kind):
    rng = np.random.default_rng(7)
    ln = rng.integers(0, 40, 150)
    if kind != "short":
        ln[{"long_first": 0, "long_middle": 70, "long_last": 149}[kind]] = 3000
    return ln


@pytest.mark.parametrize("kind", ["short", "long_first", "long_middle", "long_last"])
@pytest.mark.parametrize("heads,dk,dv,windowed", [(16, 64, 64, False), (23, 128, 40, False), (16, 64, 64, True)])
def test_gdn2_many_sequences_equal_both_layouts_bitwise(kind, heads, dk, dv, windowed, override):
    """150 sequences, some empty: the launch has the two-tile workgroups only, and
    with one long sequence among them, which is stepped a tile at a time, each
    takes two sequences.  Outputs and final states are the fixed layouts'."""
    off = np.concatenate([[0], np.cumsum(many_lengths(kind))]).astype(np.int64)
    s = W.GatedDeltaNet2Shape(1, int(off[-1]) + 3, heads, dk, dv, initial_state=False)
    inp = W.gated_deltanet2_inputs(s, seed=54)
    dev = [to_dev(inp[k]) for k in ("q", "k", "v", "g", "beta", "w")]
    start = to_dev(np.random.default_rng(8).standard_normal((150, heads, dk, dv)).astype(np.float32))
    override("gdn2_windowed", int(windowed))
    out = {}
    for ct in (0, 1, 2):
        override("gdn2_ct", ct)
        y, f = xp.gated_deltanet2_fn(*dev, start, scale=s.scale, cu_seqlens=to_dev(off), output_final_state=True)
        out[ct] = (y.cpu().numpy(), f.cpu().numpy())
        tag = [k for k in xp.last_launches() if k.startswith("Gdn2ChunkRecurKernel<")]
        assert tag and all(f",{ct},1>" in k for k in tag), xp.last_launches()
    for ct in (1, 2):
        for a, b in zip(out[0], out[ct]):
            np.testing.assert_array_equal(a, b)
    assert not out[0][0][0, off[-1]:].any()


@pytest.mark.parametrize("windowed", [False, True])
def test_gdn2_table_of_many_sequences(windowed, override):
    """700 sequences (three to a thread of the launch that builds the chunk table),
    empty ones among them, in one call and in two."""
    ln = np.random.default_rng(9).integers(0, 6, 700)
    ln[[0, 255, 256, 699]] = [0, 90, 0, 2100]
    off = np.concatenate([[0], np.cumsum(ln)]).astype(np.int64)
    s = W.GatedDeltaNet2Shape(1, int(off[-1]), 4, 64, 48, initial_state=False)
    inp = W.gated_deltanet2_inputs(s, seed=55)
    dev = [to_dev(inp[k]) for k in ("q", "k", "v", "g", "beta", "w")]
    start = to_dev(np.random.default_rng(10).standard_normal((700, 4, 64, 48)).astype(np.float32))
    override("gdn2_windowed", int(windowed))

    def call(a, b):
        y, f = xp.gated_deltanet2_fn(*(x[:, off[a]:off[b]].contiguous() for x in dev), start[a:b].contiguous(),
                                     scale=s.scale, cu_seqlens=to_dev(off[a:b + 1] - off[a]), output_final_state=True)
        return y.cpu().numpy(), f.cpu().numpy()
    y, f = call(0, 700)
    parts = [call(0, 301), call(301, 700)]
    np.testing.assert_array_equal(y, np.concatenate([x[0] for x in parts], axis=1))
    np.testing.assert_array_equal(f, np.concatenate([x[1] for x in parts]))
    np.testing.assert_array_equal(f[ln == 0], start.cpu().numpy()[ln == 0])


@pytest.mark.parametrize("offsets", [[0, 301], [1, 300], [0, 5], [296, 301], [150, 150], [301, 301], [7, 9, 250], [40, 10, 60]],
                         ids=str)
@pytest.mark.parametrize("heads,dv", [(1, 1), (1, 33), (3, 7), (4, 64)])
def test_uncovered_rows_are_zeroed(offsets, heads, dv):
    """The rows before the first sequence and behind the last (for falling offsets
    any row), over an output that held NaN, rows of odd sizes among them."""
    covered = np.zeros(301, bool)
    for lo, hi in zip(offsets, offsets[1:]):
        covered[lo:hi] = True
    cu = to_dev(np.asarray(offsets, np.int64))
    g = W.gated_deltanet2_inputs(W.GatedDeltaNet2Shape(1, 301, heads, 16, dv, initial_state=False), seed=56)
    m = W.mamba3_siso_inputs(W.Mamba3SisoShape(1, 301, heads, dv, 16), seed=57)
    for call in (xp.gated_deltanet2_fn(*(to_dev(g[k]) for k in ("q", "k", "v", "g", "beta", "w")), cu_seqlens=cu, prepare=True),
                 xp.mamba3_siso_fn(*(to_dev(m[k]) for k in ("Q", "K", "V", "ADT", "DT", "Trap", "Q_bias", "K_bias", "Angles",
                                                            "D", "Z")), cu_seqlens=cu, prepare=True)):
        out = call()
        out.fill_(float("nan"))
        out = call().cpu().numpy()
        assert not out[0, ~covered].any()
        assert np.isfinite(out).all()
