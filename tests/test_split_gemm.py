"""The grouped GEMMs on split operands (gemm_split.h) at the edges of their
tiles and at the limits of their number range."""
import os
import sys

import numpy as np
import pytest

import moe_hip as mh
import orc
from abi_types import HostMoE

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "oracle"))
import moe_backward as mb  # noqa: E402

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


# 300 experts: the general routing kernels, whose logits take 12 MB when the
# caller has no probs buffer; around 134 MB in all, with and without them.
@pytest.mark.parametrize("T", [9000, 9600, 10000, 10400])
def test_same_plan_without_probs(T):
    mh.set_expert_path(0)
    d, F, E, k = 512, 512, 300, 2
    layer = mh.Layer(d, F, E, k)
    layer.fill_synthetic(5, 0.02, 0.02)
    x, a, b, probs = (mh.DeviceArray(s) for s in ((T, d), (T, d), (T, d), (T, E)))
    mh.fill_normal_dev(x.ptr, T * d, 5, 0, 0.0, 1.0)
    layer.forward_dev(x.ptr, T, a.ptr)
    layer.forward_dev(x.ptr, T, b.ptr, probs.ptr)
    mh.synchronize()
    assert np.array_equal(a.to_host().view(np.uint32), b.to_host().view(np.uint32))
    layer.close()


def _forward(layer, x):
    T = len(x)
    dx, out = mh.DeviceArray.from_host(x), mh.DeviceArray(x.shape)
    layer.forward_dev(dx.ptr, T, out.ptr)
    mh.synchronize()
    return out.to_host()


# One expert, so that every row keeps its place.  Gate/up on 64-column tiles,
# on 256-column ones, and on those with a split tail; down in one tile column
# and in stream-K form.
@pytest.mark.parametrize("T,d,F", [(40, 64, 64), (300, 64, 8192), (700, 256, 4096)])
@pytest.mark.parametrize("value", [np.inf, np.nan])
def test_non_finite_row_leaves_others(T, d, F, value):
    """A row with a non-finite element: the other rows' bits stay."""
    layer = mh.Layer(d, F, 1, 1)
    layer.fill_synthetic(6, 0.05, 0.05)
    x = orc.synth((T, d), 8, 0, 1.0)
    ref = _forward(layer, x)
    bad = [3, T - 1]
    x[bad, 5] = value
    out = _forward(layer, x)
    assert not np.isfinite(out[bad]).any()
    rest = np.setdiff1d(np.arange(T), bad)
    assert np.array_equal(out[rest].view(np.uint32), ref[rest].view(np.uint32))
    layer.close()


# The weight gradients' tiles: 64 x 64 and 128 x 64 with two wave groups,
# 128 x 128 with one (256 rows per expert and more).
@pytest.mark.parametrize("T,d,F,E", [(200, 64, 64, 2), (1000, 256, 1024, 8), (2048, 512, 2048, 8)])
def test_non_finite_gradient_leaves_others(T, d, F, E):
    """An infinity in one element of dout: the infinities that float products
    make of it in its column of dW_down, and the bits of the other columns and
    of the other rows' dx stay."""
    layer = mh.Layer(d, F, E, 1)
    layer.fill_synthetic(6, 0.05, 0.05)
    x, dout = orc.synth((T, d), 9, 0, 1.0), orc.synth((T, d), 9, 1, 1.0)
    dxd, ids = mh.DeviceArray.from_host(x), mh.DeviceArray((T, 1), np.int32)
    out = mh.DeviceArray((T, d))
    layer.forward_dev(dxd.ptr, T, out.ptr, None, ids.ptr)
    res = []
    for value in (dout[7, 9], np.inf):
        dout[7, 9] = value
        outs = [mh.DeviceArray(s) for s in ((T, d), (d, E), (E, d, F), (E, d, F), (E, F, d))]
        dod = mh.DeviceArray.from_host(dout)
        layer.backward_dev(dxd.ptr, T, dod.ptr, 0.0, *[a.ptr for a in outs])
        mh.synchronize()
        res.append((outs[0].to_host(), outs[4].to_host()))
    (dx0, dw0), (dx1, dw1) = res
    e = int(ids.to_host()[7, 0])
    col = dw1[e][:, 9].copy()
    wg, wu = layer.get_expert(e)[:2]
    g, u = (x[7].astype(np.float64) @ w.astype(np.float64) for w in (wg, wu))
    assert np.array_equal(col, np.sign(g * u) * np.inf)
    assert not np.isfinite(dx1[7]).any()
    dw1[e][:, 9], dx1[7] = dw0[e][:, 9], dx0[7]
    assert np.array_equal(dw0.view(np.uint32), dw1.view(np.uint32))
    assert np.array_equal(dx0.view(np.uint32), dx1.view(np.uint32))
    layer.close()


# The operands' range goes down to the smallest floats.  Gate sums see only the
# scaled half of a row, up sums the other half, so H (and the down sums) take
# the scale once; W_down is raised to bring the outputs back among the normal
# floats.
@pytest.mark.parametrize("T,d,F", [(40, 64, 64), (700, 256, 512)])
@pytest.mark.parametrize("e", [70, 90, 109, 118, 125])
def test_small_operands(T, d, F, e):
    hw = _layer(d, F, 2, 1, 11)
    x = orc.synth((T, d), 6, 0, 1.0)
    x[:, d // 2:] *= np.float32(2.0 ** -e)
    hw.wg[:, :d // 2] = 0
    hw.wu[:, d // 2:] = 0
    hw.wd *= np.float32(2.0 ** 24)
    out, probs, ids = mh.moe_forward(x, hw)
    # (x * 2^-125 has subnormal elements, exact to 2^-149: they enter the
    # reference as rounded; bound as in test_tile_edges)
    assert orc.rel_l2(out, _layer64(x, hw, ids, probs)) < 3e-6


@pytest.mark.parametrize("e", [90, 115, 118])
@pytest.mark.parametrize("T,d,F", [(200, 128, 192), (90, 64, 64)])
def test_small_gradients(T, d, F, e):
    """Gradients of a loss scaled by 2^-e, to the precision of an unscaled one."""
    r = np.random.default_rng(T)
    f = lambda *s: (0.3 * r.standard_normal(s)).astype(np.float32)
    hw = HostMoE(f(d, 4), f(4, d, F), f(4, d, F), f(4, F, d), 2)
    x, dout = orc.synth((T, d), 7, 0, 1.0), orc.synth((T, d), 7, 1, 1.0)
    ids = orc.route(x, hw.wr, 2)[1]
    g = mb.moe_backward64(x, hw.wr, hw.wg, hw.wu, hw.wd, ids, dout)
    layer = mh.Layer(d, F, 4, 2)
    layer.load(hw)
    outs = dict(dx=mh.DeviceArray((T, d)), dwr=mh.DeviceArray((d, 4)), dwg=mh.DeviceArray((4, d, F)),
                dwu=mh.DeviceArray((4, d, F)), dwd=mh.DeviceArray((4, F, d)))
    dxd, dod = mh.DeviceArray.from_host(x), mh.DeviceArray.from_host(dout * np.float32(2.0 ** -e))
    layer.backward_dev(dxd.ptr, T, dod.ptr, 0.0, *[a.ptr for a in outs.values()])
    mh.synchronize()
    for name, a in outs.items():
        # Chains of up to four sums of at most 192 products each and the
        # SwiGLU's derivative: under 3e-6 (as above).
        assert orc.rel_l2(a.to_host().astype(np.float64) * 2.0 ** e, g[name]) < 3e-6, name
    layer.close()


# Widths past 1024 that 256 does not divide: gate/up's last 256-column tile
# reaches past N (64 features of its 128 here; with 12 experts 96 of 128).
@pytest.mark.parametrize("T,d,F,E,k", [(700, 64, 5440, 2, 1), (1003, 320, 1376, 12, 3)])
def test_wide_tiles_past_the_width(T, d, F, E, k):
    hw = _layer(d, F, E, k, T)
    x = orc.synth((T, d), 12, 0, 1.0)
    out, probs, ids = mh.moe_forward(x, hw)
    # (as in test_tile_edges, the down sums up to 5440 products long)
    assert orc.rel_l2(out, _layer64(x, hw, ids, probs)) < 4e-6


# gate/up on 256-column tiles (one wave for 128 rows, last m-tiles of one to
# four 32-row blocks), without and with a split tail (2 and 4 pieces).
@pytest.mark.parametrize("T,d,F", [(330, 64, 6656), (300, 64, 6656), (700, 64, 5632), (700, 128, 5632)])
@pytest.mark.parametrize("where", ["gate", "up", "down"])
@pytest.mark.parametrize("value", [np.inf, np.nan, 3.4e38])
def test_limits_wide_tiles(T, d, F, where, value):
    test_limits(T, d, F, where, value)


def _backward64(x, dout, wg, wu, wd, ids):
    """dx and the experts' gradients of a top-1 layer (gate weights 1, no
    router gradient) in float64."""
    dx = np.zeros(x.shape)
    dw = []
    for e in range(len(wg)):
        t = np.nonzero(ids[:, 0] == e)[0]
        xe, dy, g, u, d = (a.astype(np.float64) for a in (x[t], dout[t], wg[e], wu[e], wd[e]))
        g, u, wge, wue = xe @ g, xe @ u, g, u
        s = 1 / (1 + np.exp(-g))
        dh = dy @ d.T
        dg, du = dh * u * (s + g * s * (1 - s)), dh * g * s
        dx[t] = dg @ wge.T + du @ wue.T
        dw.append((xe.T @ dg, xe.T @ du, (g * s * u).T @ dy))
    return dx, *(np.stack(w) for w in zip(*dw))


# The weight gradients' tiles at hundreds of rows per expert: 128 x 64 with two
# wave groups, 128 x 128 with one (512 tiles and more), and both at expert
# loads that leave part of a round of steps (16 rows, or 32 with two groups).
@pytest.mark.parametrize("T,d,F,E", [(1000, 256, 1024, 8), (1111, 256, 1024, 8), (2048, 512, 2048, 8), (1777, 512, 2048, 8)])
def test_weight_gradients(T, d, F, E):
    layer = mh.Layer(d, F, E, 1)
    layer.fill_synthetic(13, 0.05, 0.05)
    x, dout = orc.synth((T, d), 13, 0, 1.0), orc.synth((T, d), 13, 1, 1.0)
    dxd, ids, out = mh.DeviceArray.from_host(x), mh.DeviceArray((T, 1), np.int32), mh.DeviceArray((T, d))
    layer.forward_dev(dxd.ptr, T, out.ptr, None, ids.ptr)
    outs = [mh.DeviceArray(s) for s in ((T, d), (d, E), (E, d, F), (E, d, F), (E, F, d))]

    def run(dout):
        dod = mh.DeviceArray.from_host(dout)
        layer.backward_dev(dxd.ptr, T, dod.ptr, 0.0, *[a.ptr for a in outs])
        mh.synchronize()
        return [a.to_host() for a in (outs[0], *outs[2:])]

    got = run(dout)
    w = [np.stack(m) for m in zip(*(layer.get_expert(e) for e in range(E)))]
    ids = ids.to_host()
    ref = _backward64(x, dout, *w, ids)
    for a, b in zip(got, ref):
        assert orc.rel_l2(a, b) < 3e-6   # (sums of at most 4096 products, as above)
    # One infinity in dout: its row of dH, dG and dU is infinite, and so are
    # the sums of the expert's gradients that take it.
    dout[7, 9] = np.inf
    bad = run(dout)
    e = int(ids[7, 0])
    wg, wu, wd = (m[e].astype(np.float64) for m in w)
    g, u = x[7].astype(np.float64) @ wg, x[7].astype(np.float64) @ wu
    s = 1 / (1 + np.exp(-g))
    sign = np.sign(wd[:, 9])
    inf = lambda a, b: np.sign(np.outer(a, b)) * np.inf
    assert np.array_equal(bad[1][e], inf(x[7], sign * u * (s + g * s * (1 - s))))
    assert np.array_equal(bad[2][e], inf(x[7], sign * g * s))
    assert np.array_equal(bad[3][e][:, 9], inf(g * s * u, [1.0])[:, 0])
    assert np.isfinite(np.delete(bad[3][e], 9, 1)).all()
    for a, b in zip(bad[1:], got[1:]):
        assert np.array_equal(np.delete(a, e, 0).view(np.uint32), np.delete(b, e, 0).view(np.uint32))
    layer.close()


# Experts with few rows (none, one, and up to a few steps of 16 past what the
# short form's mean allows), on every tile: 64 x 64, 128 x 64 (both widths),
# 128 x 128, with one and two wave groups.
@pytest.mark.parametrize("d,F,E", [(64, 64, 5), (192, 128, 12), (128, 448, 60), (448, 128, 60), (256, 1024, 20), (512, 512, 40)])
@pytest.mark.parametrize("T", [1, 17, 100])
def test_weight_gradients_few_rows(T, d, F, E):
    layer = mh.Layer(d, F, E, 1)
    layer.fill_synthetic(15, 0.3, 0.05)
    layer.set_bias((3.0 * np.cos(np.arange(E))).astype(np.float32))   # (uneven loads)
    x, dout = orc.synth((T, d), 15, 0, 1.0), orc.synth((T, d), 15, 1, 1.0)
    dxd, dod, ids, out = mh.DeviceArray.from_host(x), mh.DeviceArray.from_host(dout), mh.DeviceArray((T, 1), np.int32), mh.DeviceArray((T, d))
    layer.forward_dev(dxd.ptr, T, out.ptr, None, ids.ptr)
    outs = [mh.DeviceArray(s) for s in ((T, d), (d, E), (E, d, F), (E, d, F), (E, F, d))]
    layer.backward_dev(dxd.ptr, T, dod.ptr, 0.0, *[a.ptr for a in outs])
    mh.synchronize()
    w = [np.stack(m) for m in zip(*(layer.get_expert(e) for e in range(E)))]
    ref = _backward64(x, dout, *w, ids.to_host())
    for a, b in zip((outs[0], *outs[2:]), ref):
        assert orc.rel_l2(a.to_host(), b) < 3e-6   # (as in test_weight_gradients)
    layer.close()


# The down projection's tiles whole (K = 96), in even pieces (of two slices; of
# four; bounded by a token's slots) and in runs that touch
# two tiles (counted on the most and on the fewest tiles).
@pytest.mark.parametrize("T,d,F,E,k", [(60, 192, 96, 30, 6), (97, 128, 192, 3, 3), (118, 256, 256, 1, 1), (621, 256, 2304, 2, 1), (24, 256, 3200, 8, 6),
                                       (1500, 512, 512, 4, 2), (900, 640, 1056, 6, 3), (129, 1024, 4096, 1, 1)])
def test_down_projection_pieces(T, d, F, E, k):
    hw = _layer(d, F, E, k, T)
    x = orc.synth((T, d), 16, 0, 1.0)
    out, probs, ids = mh.moe_forward(x, hw)
    assert orc.rel_l2(out, _layer64(x, hw, ids, probs)) < 3e-6   # (as in test_tile_edges)
