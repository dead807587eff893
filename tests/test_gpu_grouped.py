"""The expert-grouped f16 kernels past 16 tokens and in short prefills: against
the per-assignment GEMVs on the same weights, at the edges of their ranges
(groups of 4, one-launch routing up to 64 tokens, partly filled units of 8
tiles) and with scales that f16 terms cannot carry; and which calls take them."""
import numpy as np
import pytest

from conftest import rel_l2, say
from midge_amd import DevBuf, device, synth
from midge_amd.moe import MoELayer, Stack, expert_major_dev, moe_dev, moe_prefill, moe_prefill_dev
from midge_amd.synth import Keys, MoEShape
from oracle import pyoracle as po

pytestmark = pytest.mark.gpu
# A layer's update from inputs held to 2^-22 of each column's largest value and
# f32 sums in another order: 2e-6 of x per token (as test_gpu_moe's SPLIT_TOL).
TOL = 2e-6
MID = MoEShape(hidden=256, ffn=192, n_experts=64, top_k=4)
WIDE = MoEShape(hidden=1536, ffn=1088, n_experts=32, top_k=2)   # ffn / 4 and hidden / 8 leave partial units
SMALL = MoEShape(hidden=64, ffn=64, n_experts=130, top_k=16)


def make(shape, seed, scales="plain", bias=None):
    keys = Keys(seed)
    ex = synth.host_layer_experts(shape, keys, 0).copy()
    if scales != "plain":
        # expert 1: every gate scale; expert 2: one down scale of the last row
        val = {"odd": 1.37, "big": 2.0 ** 14, "tiny": 2.0 ** -24, "zero": 0.0, "subnormal": 2.0 ** -20}[scales]
        v = np.frombuffer(np.float16(val).tobytes(), np.uint8)
        lay = shape.layout
        g0 = lay.offset(0, 1, 0, 1)
        ex[g0:g0 + 2 * shape.ffn * (shape.hidden // 32)] = np.tile(v, shape.ffn * (shape.hidden // 32))
        d0 = lay.offset(0, 2, 2, 1) + 2 * (shape.hidden * (shape.ffn // 32) - 1)
        ex[d0:d0 + 2] = v
    w, s, b, nw = synth.host_router(shape, keys, 0)
    if bias is not None:
        b = bias(b)
    return keys, (ex, w, s, b, nw), MoELayer.host(shape, ex, w, s, b, nw)


@pytest.mark.parametrize("shape,n,scales", [
    (MID, 2, "plain"), (MID, 64, "plain"), (MID, 65, "plain"), (MID, 127, "plain"), (WIDE, 33, "plain"),
    (SMALL, 3, "plain"), (SMALL, 64, "plain"),
    (MID, 60, "odd"), (MID, 60, "big"), (MID, 60, "tiny"), (MID, 60, "zero"), (MID, 60, "subnormal"), (WIDE, 70, "odd"),
], ids=lambda v: v if isinstance(v, (int, str)) else f"{v.hidden}x{v.ffn}e{v.n_experts}")
def test_short_prefill(mh, path_switch, shape, n, scales):
    say(f"short prefill {shape.hidden}x{shape.ffn} E={shape.n_experts} n={n} scales={scales}")
    path_switch("GROUPED")
    keys, arrays, lay = make(shape, 11, scales)
    X = synth.host_x(shape, keys, n, step=2)
    xg, selg, wg = moe_prefill(lay, X)
    path_switch("NO_MFMA")
    xv, selv, wv = moe_prefill(lay, X)
    xr, selr, _ = po.moe_prefill(po.layer_struct(shape, *arrays), X)
    lay.release()
    assert (selg == selv).all() and (selg == selr).all()
    assert not np.array_equal(xg, xv)   # the matrix cores ran
    for t in range(n):
        assert rel_l2(xg[t], xv[t]) < TOL, t
    assert rel_l2(xg, xr) < 1e-4


@pytest.mark.parametrize("shape,n,unfilled", [(MID, 17, False), (MID, 64, False), (MID, 65, True), (WIDE, 40, False),
                                              (SMALL, 50, True)],
                         ids=lambda v: f"{v.hidden}x{v.ffn}e{v.n_experts}" if isinstance(v, MoEShape) else str(v))
def test_stack_many_tokens(mh, path_switch, shape, n, unfilled):
    say(f"stack decode {shape.hidden}x{shape.ffn} E={shape.n_experts} n={n} unfilled={unfilled}")

    def bias(b):
        b = np.full_like(b, -1e31)
        b[[2, 11]] = 0.0
        return b

    path_switch("GROUPED")
    keys, arrays, lay = make(shape, 12, bias=bias if unfilled else None)
    X, k = synth.host_x(shape, keys, n, step=1), shape.top_k
    st = Stack([lay], max_batch=n)
    out = []
    for gemv in (False, True):
        path_switch("BATCH_GEMV", gemv)
        xd, sd, ud = DevBuf.from_array(X), DevBuf(4 * n * k), DevBuf.from_array(np.zeros(shape.n_experts, np.uint32))
        st.decode(xd, n, sd, usage=ud)
        mh.sync()
        out.append((xd.download(np.float32, X.shape), sd.download(np.int32, (n, k)),
                    ud.download(np.uint32, (shape.n_experts,))))
        for d in (xd, sd, ud):
            d.free()
    st.destroy()
    lay.release()
    (xg, sg, ug), (xv, sv, uv) = out
    assert (sg == sv).all() and (ug == uv).all()
    assert (ug == np.bincount(sg[sg >= 0], minlength=shape.n_experts)).all()
    assert not np.array_equal(xg, xv)
    for t in range(n):
        assert rel_l2(xg[t], xv[t]) < TOL, t
    if unfilled:
        assert (sg[:, 2:] == -1).all()


def test_given_routing_with_unroutable_slots(mh, path_switch):
    """mh_expert_major_dev takes any selection: slots outside [0, E) add nothing."""
    shape, n = MID, 40
    say("expert major, unroutable slots")
    path_switch("GROUPED")
    keys, arrays, lay = make(shape, 13)
    X = synth.host_x(shape, keys, n, step=4)
    rng = np.random.default_rng(5)
    sel = rng.integers(-2, shape.n_experts + 2, (n, shape.top_k)).astype(np.int32)
    sel[7] = -1
    w = rng.random((n, shape.top_k)).astype(np.float32)
    out = []
    for gemv in (False, True):
        path_switch("NO_MFMA", gemv)
        bufs = [DevBuf.from_array(a) for a in (X, sel, w, X)]
        expert_major_dev(lay, n, *bufs)
        mh.sync()
        out.append(bufs[3].download(np.float32, X.shape))
        for d in bufs:
            d.free()
    lay.release()
    assert np.array_equal(out[0][7], X[7])
    for t in range(n):
        assert rel_l2(out[0][t], out[1][t]) < TOL, t


@pytest.mark.parametrize("kind,n,grouped", [("prefill", 2, False), ("prefill", 8, False), ("prefill", 63, True),
                                            ("experts", 8, False), ("experts", 48, True), ("moe", 2, False),
                                            ("moe", 8, False), ("moe", 64, True), ("stack", 16, True), ("stack", 17, True),
                                            ("stack", 64, True)])
def test_route(mh, path_switch, kind, n, grouped):
    """Few assignments of a small layer run on the GEMVs, many on the grouped
    kernels (a scanned stack's up to 64 assignments in any case); where the
    GEMVs run, the result is theirs bit for bit."""
    shape, k = MoEShape(hidden=1024, ffn=768, n_experts=32, top_k=4), 4
    say(f"route {kind} n={n}")
    keys, arrays, lay = make(shape, 14)
    X = synth.host_x(shape, keys, n, step=1)
    rng = np.random.default_rng(n)
    sel = np.argsort(rng.random((n, shape.n_experts)), axis=1)[:, :k].astype(np.int32)
    w = np.full((n, k), 0.25, np.float32)
    st = Stack([lay], max_batch=64) if kind == "stack" else None
    out = []
    for gemv in (False, True):
        path_switch("NO_MFMA" if kind in ("prefill", "experts") else "BATCH_GEMV", gemv)
        xd, xb, sd, wd = (DevBuf.from_array(a) for a in (X, X, sel, w))
        device.profile_enable()
        device.profile_reset()
        if kind == "prefill":
            moe_prefill_dev(lay, xd, n, sd, wd)
        elif kind == "experts":
            expert_major_dev(lay, n, xb, sd, wd, xd)
        elif kind == "moe":
            moe_dev(lay, xd, n, sd, wd)
        else:
            st.decode(xd, n, sd, wd)
        mh.sync()
        ran = device.profile_query("grouped_gu")[1], device.profile_query("expert_gu")[1]
        device.profile_enable(False)
        assert ran == ((0, 1) if gemv or not grouped else (1, 0))
        out.append(xd.download(np.float32, X.shape))
        for d in (xd, xb, sd, wd):
            d.free()
    if st:
        st.destroy()
    lay.release()
    if grouped:
        assert max(rel_l2(a, b) for a, b in zip(*out)) < TOL
    else:
        assert np.array_equal(*out)


@pytest.mark.parametrize("scales", ["plain", "odd"])
def test_values_that_are_not_finite(mh, path_switch, scales):
    """Inputs with infinities, NaN, f32's largest and subnormal numbers: the same
    infinities and NaN as the GEMVs' f32 sums give, the same bits for the tokens
    beside them as without them, and subnormal inputs lost without a trace."""
    shape, n = MID, 24
    say(f"grouped, values that are not finite, scales={scales}")
    path_switch("GROUPED")
    keys, arrays, lay = make(shape, 15, scales)
    X = synth.host_x(shape, keys, n, step=1)
    plain = X.copy()
    X[1, 5] = np.inf
    X[4, 200] = -np.inf
    X[7, [0, 255]] = np.inf, -np.inf
    X[9, 31] = np.nan
    X[12, 64] = np.nan
    X[12, 3] = np.inf
    X[15] *= 1e30          # large, finite sums
    X[18] *= 1e-42         # subnormal
    X[20] = 0.0
    odd = [1, 4, 7, 9, 12, 15, 18, 20]
    rng = np.random.default_rng(6)
    sel = rng.integers(0, 6, (n, shape.top_k)).astype(np.int32)   # groups that odd and plain tokens share
    w = rng.uniform(0.5, 1.0, (n, shape.top_k)).astype(np.float32)
    out = []
    for x, gemv in ((X, False), (X, True), (plain, False)):
        path_switch("NO_MFMA", gemv)
        bufs = [DevBuf.from_array(a) for a in (x, sel, w, np.zeros_like(X))]
        expert_major_dev(lay, n, *bufs)
        mh.sync()
        out.append(bufs[3].download(np.float32, X.shape))
        for d in bufs:
            d.free()
    lay.release()
    got, want, alone = out
    assert not np.isfinite(want[[1, 4, 7, 9, 12]]).all()
    assert (np.isnan(got) == np.isnan(want)).all() and (np.isposinf(got) == np.isposinf(want)).all()
    assert (np.isneginf(got) == np.isneginf(want)).all()
    rest = np.setdiff1d(np.arange(n), odd)
    assert np.array_equal(got[rest], alone[rest])
    for t in list(rest) + [15, 18, 20]:
        assert np.isfinite(want[t]).all() and rel_l2(got[t], want[t]) < TOL, t


def experts_f64(shape, ex, xb, sel, w):
    """sum_i w_i expert_{sel_i}(xb) per token in 64 bits, from the layer's bytes."""
    lay, out = shape.layout, np.zeros(xb.shape)
    code = np.array([0, 0.5, 1, 1.5, 2, 3, 4, 6, 0, -0.5, -1, -1.5, -2, -3, -4, -6])

    def matrix(e, m):
        rows, cols = lay.rows[m], lay.cols[m]
        q = ex[lay.offset(0, e, m, 0):][:rows * cols // 2].reshape(rows, -1)
        sc = ex[lay.offset(0, e, m, 1):][:rows * cols // 16].view(np.float16).astype(np.float64).reshape(rows, -1)
        b = ex[lay.offset(0, e, m, 2):][:4 * rows].view(np.float32).astype(np.float64)
        v = np.stack((code[q & 15], code[q >> 4]), -1).reshape(rows, cols // 32, 32)
        return (v * sc[:, :, None]).reshape(rows, cols), b

    for e in np.unique(sel):
        t, i = np.nonzero(sel == e)
        (wg, bg), (wu, bu), (wd, bd) = (matrix(e, m) for m in range(3))
        x = xb[t].astype(np.float64)
        g, u = np.minimum(x @ wg.T + bg, shape.limit), np.clip(x @ wu.T + bu, -shape.limit, shape.limit)
        h = g / (1 + np.exp(-shape.alpha * g)) * (u + 1)
        np.add.at(out, t, (h @ wd.T + bd) * w[t, i, None].astype(np.float64))
    return out


@pytest.mark.parametrize("hidden,ffn", [(256, 192), (512, 2048), (1024, 768), (2880, 2880)])
def test_error_against_64_bits(mh, path_switch, hidden, ffn):
    """The grouped kernels hold an input to 23 bits (two f16 terms) where the
    GEMVs have f32's 24, and add in longer chains of the matrix core where those
    add lane by lane: their outputs are no further from 64 bits."""
    shape = MoEShape(hidden=hidden, ffn=ffn, n_experts=4, top_k=2)
    say(f"grouped error {hidden}x{ffn}")
    path_switch("GROUPED")
    keys, (ex, *_), lay = make(shape, 16)
    n = 15   # fewer than 8 assignments per expert
    rng = np.random.default_rng(hidden)
    err = []
    for rep in range(4):
        xb = rng.standard_normal((n, hidden)).astype(np.float32)
        sel = np.argsort(rng.random((n, 4)), axis=1)[:, :2].astype(np.int32)
        w = rng.uniform(0.2, 0.8, (n, 2)).astype(np.float32)
        want = experts_f64(shape, ex.view(np.uint8).ravel(), xb, sel, w)
        for gemv in (False, True):
            path_switch("NO_MFMA", gemv)
            bufs = [DevBuf.from_array(a) for a in (xb, sel, w, np.zeros_like(xb))]
            expert_major_dev(lay, n, *bufs)
            mh.sync()
            err.append(rel_l2(bufs[3].download(np.float32, xb.shape), want))
            for d in bufs:
                d.free()
    lay.release()
    grouped, gemv = np.sqrt(np.mean(np.square(err[0::2]))), np.sqrt(np.mean(np.square(err[1::2])))
    say(f"grouped {grouped:.3g}, GEMVs {gemv:.3g}")
    assert grouped < 1.02 * gemv < 4e-7
