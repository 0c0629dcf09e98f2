"""The grouped GEMMs on split operands (gemm_split.h) at the edges of their
tiles and at the limits of their number range."""
import numpy as np
import pytest

import moe_hip as mh
import orc
from abi_types import HostMoE

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _grouped():
    mh.check(mh.lib().moe_hip_init(0))
    mh.set_expert_path(1)
    yield
    mh.set_expert_path(0)


def _layer(d, F, E, k, seed):
    r = np.random.default_rng(seed)
    f = lambda *s: (0.05 * r.standard_normal(s)).astype(np.float32)
    return HostMoE(f(d, E), f(E, d, F), f(E, d, F), f(E, F, d), k)


def _layer64(x, hw, ids, probs):
    """The layer of the routed rows in float64 (routing as given)."""
    out = np.zeros(x.shape)
    sel = np.take_along_axis(probs.astype(np.float64), ids, 1)
    gw = sel / sel.sum(1, keepdims=True)
    with np.errstate(all="ignore"):
        for e in range(hw.E):
            t, s = np.nonzero(ids == e)
            xe = x[t].astype(np.float64)
            g, u = xe @ hw.wg[e].astype(np.float64), xe @ hw.wu[e].astype(np.float64)
            np.add.at(out, t, gw[t, s][:, None] * ((g / (1 + np.exp(-g)) * u) @ hw.wd[e].astype(np.float64)))
    return out


# Rows around the 32-row blocks and 128-row tiles (one expert takes all with
# E = 1), widths that leave waves of the last column tile without columns,
# and reductions of one and of many 32-wide slices.
@pytest.mark.parametrize("T", [1, 31, 33, 64, 96, 127, 128, 129, 257])
@pytest.mark.parametrize("d,F", [(64, 32), (64, 96), (192, 160), (320, 256), (512, 288)])
def test_tile_edges(T, d, F):
    hw = _layer(d, F, 1, 1, T + d)
    x = orc.synth((T, d), 3, 0, 1.0)
    out, probs, ids = mh.moe_forward(x, hw)
    ref = _layer64(x, hw, ids, probs)
    # Each output carries two sums of d and one of F products; a running
    # float sum of n terms is off by about sqrt(n) 2^-25 of its size, and the
    # SwiGLU by 2 ulp: under 3e-6 at these widths.
    assert orc.rel_l2(out, ref) < 3e-6


@pytest.mark.parametrize("E,k,T", [(3, 2, 300), (8, 2, 1000), (40, 8, 200)])
def test_several_experts(E, k, T):
    hw = _layer(256, 320, E, k, E)
    x = orc.synth((T, 256), 4, 0, 1.0)
    out, probs, ids = mh.moe_forward(x, hw)
    assert orc.rel_l2(out, _layer64(x, hw, ids, probs)) < 3e-6


@pytest.mark.parametrize("T,d,F", [(5, 64, 64), (200, 320, 96), (130, 256, 512)])
@pytest.mark.parametrize("where", ["gate", "up", "down"])
@pytest.mark.parametrize("value", [np.inf, -np.inf, np.nan, 3.4e38])
def test_limits(T, d, F, where, value):
    """An infinity, a NaN and a float above the largest bfloat16 among the
    weights: the outputs are infinite, NaN and finite where float products
    make them so."""
    hw = _layer(d, F, 2, 1, 9)
    x = orc.synth((T, d), 5, 0, 1.0)
    {"gate": hw.wg, "up": hw.wu, "down": hw.wd}[where][0, 7, 11] = value
    if value == 3.4e38:
        x[:, 7] *= 1e-36    # (finite products)
    out, probs, ids = mh.moe_forward(x, hw)
    ref = _layer64(x, hw, ids, probs)
    if value == 3.4e38 and where == "down":
        ref = np.where(np.abs(ref) > np.finfo(np.float32).max, np.sign(ref) * np.inf, ref)
    assert np.array_equal(np.isnan(out), np.isnan(ref))
    assert np.array_equal(np.isposinf(out), np.isposinf(ref))
    assert np.array_equal(np.isneginf(out), np.isneginf(ref))
    fin = np.isfinite(ref)
    # (3e-6 of the norm, as above; one output may cancel terms of the large
    # feature, so single elements have no relative bound)
    assert orc.rel_l2(out[fin], ref[fin]) < 3e-6


# Layers whose temporaries fit the allocation-free entry point's scratch only
# without the split tail, and only without split sums.
@pytest.mark.parametrize("T,d,F,E,k", [(4096, 512, 2048, 8, 2), (6000, 320, 1376, 12, 3), (1003, 320, 1376, 12, 3)])
def test_same_plan_without_allocation(T, d, F, E, k):
    mh.set_expert_path(0)
    layer = mh.Layer(d, F, E, k)
    layer.fill_synthetic(5, 0.02, 0.02)
    x, a, b = (mh.DeviceArray((T, d)) for _ in range(3))
    mh.fill_normal_dev(x.ptr, T * d, 5, 0, 0.0, 1.0)
    layer.forward_dev(x.ptr, T, a.ptr)
    layer.forward_dev_noalloc(x.ptr, T, b.ptr)
    mh.synchronize()
    assert np.array_equal(a.to_host().view(np.uint32), b.to_host().view(np.uint32))
    layer.close()
