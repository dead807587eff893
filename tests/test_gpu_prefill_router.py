"""The routers of several tokens: which one a call takes (k_combine_route,
k_route_tokens or three launches) and that its choice, weights and outputs are
those of the three launches, over the token counts, widths and expert counts at
the edges of their rules and tiles."""
import numpy as np
import pytest

from conftest import rel_l2, say
from midge_amd import DevBuf, _lib, device, synth
from midge_amd.moe import MoELayer, Stack, moe_prefill_dev
from midge_amd.synth import Keys, MoEShape

pytestmark = pytest.mark.gpu


def make(hidden, experts, top_k=2, seed=31, **kw):
    shape = MoEShape(hidden=hidden, ffn=64, n_experts=experts, top_k=top_k, **kw)
    keys = Keys(seed)
    w, s, b, nw = synth.host_router(shape, keys, 0)
    # (a tenth of the router's scales: logits of a few units, whose softmax
    # does not hide the f32 sums' differences)
    return shape, keys, MoELayer.host(shape, synth.host_layer_experts(shape, keys, 0), w, s * np.float32(0.1), b, nw)


def launched(names):
    return [device.profile_query(n)[1] for n in names]


@pytest.mark.parametrize("kind,hidden,experts,n,want", [
    ("prefill", 256, 128, 64, "combine_route"), ("prefill", 256, 130, 64, "topk"), ("prefill", 256, 1024, 8, "combine_route"),
    ("prefill", 256, 1024, 9, "topk"), ("prefill", 2880, 256, 64, "combine_route"), ("prefill", 64, 64, 65, "route_tokens"),
    ("prefill", 256, 128, 300, "topk"), ("prefill", 512, 128, 65, "topk"), ("prefill", 512, 128, 100, "route_tokens"),
    ("prefill", 1024, 520, 97, "topk"), ("prefill", 1024, 520, 98, "route_tokens"), ("stack", 256, 512, 16, "combine_route"),
    ("stack", 256, 512, 17, "topk"), ("stack", 256, 128, 64, "combine_route")])
def test_router_choice(mh, kind, hidden, experts, n, want):
    say(f"router choice {kind} {hidden} E={experts} n={n}")
    shape, keys, lay = make(hidden, experts)
    xd = DevBuf.from_array(synth.host_x(shape, keys, n, step=1))
    st = Stack([lay], max_batch=64) if kind == "stack" else None
    names = ["combine_route", "route_tokens", "topk"]
    device.profile_enable()
    device.profile_reset()
    if st:
        st.decode(xd, n)
    else:
        moe_prefill_dev(lay, xd, n)
    mh.sync()
    ran = launched(names)
    device.profile_enable(False)
    if st:
        st.destroy()
    xd.free()
    lay.release()
    assert ran == [int(v == want) for v in names]


# Per token, the outputs of two prefills whose normed inputs differ in their
# last bits: each holds them within the matrix product's bound (6.2e-4, as in
# test_gpu_prefill_gemm), so they differ by at most sqrt(2) of it. An input
# block that went wrong would show as 1 / sqrt(blocks) >= 0.1.
GEMM_TOL = 8.8e-4
# Weights: logits of |l| < 16 as f32 sums in two orders (1e-6 of them apart).
WTOL = dict(rtol=1.6e-5, atol=1e-7)
F32_TOL = 2e-5   # the f32 paths: the weights', and twice the grouped kernels' 2e-6


@pytest.mark.parametrize("hidden,experts,n,kw", [
    # records: one to three chunks a lane, odd lanes' blocks, half and whole last K steps
    (64, 4, 66, {}), (1024, 4, 66, {}), (1088, 4, 130, {}), (2112, 4, 67, {}), (2880, 4, 130, {}), (3072, 4, 65, {}),
    # waves per token: 8, 4, 2, 1, and a last block of fewer tokens
    (64, 4, 511, {}), (64, 4, 512, {}), (2112, 4, 513, {}), (64, 4, 1023, {}), (128, 4, 1025, {}), (64, 4, 2047, {}),
    (192, 4, 2048, {}), (1088, 4, 2049, {}),
    # experts: not a multiple of four, more than 128 and than 256
    (64, 7, 65, {}), (1024, 130, 130, {}), (1024, 257, 120, {}), (1024, 130, 600, {}), (512, 257, 2050, {}),
    # softmax over all logits; f32 rows (other experts, widths that no matrix product takes, few tokens per expert)
    (256, 8, 100, dict(router_norm=0)), (1056, 8, 70, {}), (256, 8, 70, dict(expert_dt=_lib.DT_Q4G32)), (2880, 64, 70, {})])
def test_route_tokens(mh, path_switch, hidden, experts, n, kw):
    """Against the three launches on the same tokens: the same choice, its
    weights, and outputs within the paths' bounds; x, and in one run the norm's
    weights, on a 4-byte boundary give the same bits as on a 16-byte one."""
    say(f"route tokens {hidden} E={experts} n={n} {kw}")
    shape, keys, lay = make(hidden, experts, **kw)
    X = synth.host_x(shape, keys, n, step=2)
    w, s, b, nw = synth.host_router(shape, keys, 0)
    nwd = DevBuf.from_array(np.concatenate([nw[:1], nw]).astype(np.float32))
    out = []
    for mode in ("one", "shifted", "split"):
        path_switch("SPLIT_ROUTE", mode == "split")
        xd = DevBuf.from_array(np.concatenate([X.ravel()[:1], X.ravel()]))
        x0 = DevBuf.from_array(X)
        sd, wd = DevBuf(4 * n * 2), DevBuf(4 * n * 2)
        norm = lay.mlp_norm
        if mode == "shifted":
            lay.mlp_norm = nwd.ptr + 4
        device.profile_enable()
        device.profile_reset()
        moe_prefill_dev(lay, xd.ptr + 4 if mode == "shifted" else x0, n, sd, wd)
        mh.sync()
        assert launched(["route_tokens"])[0] == (mode != "split")
        device.profile_enable(False)
        lay.mlp_norm = norm
        x = xd.download(np.float32, (X.size,), offset=4).reshape(X.shape) if mode == "shifted" \
            else x0.download(np.float32, X.shape)
        out.append((x - X, sd.download(np.int32, (n, 2)), wd.download(np.float32, (n, 2))))
        for d in (xd, x0, sd, wd):
            d.free()
    nwd.free()
    gemm = shape.expert_dt == _lib.DT_MXFP4 and hidden % 64 == 0 and 2 * n >= 8 * experts
    lay.release()
    (dx, sel, wt), shifted, (dv, sv, wv) = out
    assert (sel == sv).all() and np.allclose(wt, wv, **WTOL)
    assert all(np.array_equal(a, b) for a, b in zip(shifted, out[0]))
    tol = GEMM_TOL if gemm else F32_TOL
    worst = max(rel_l2(dx[t], dv[t]) for t in range(n))
    say(f"worst token {worst:.3g}")
    assert worst < tol
