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
