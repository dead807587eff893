"""The scaled-matrix-core prefill at the edges of its tiles (32 rows and tokens,
passes of up to 2 token tiles, K steps of 128 columns, blocks of 128 rows)
against the per-assignment GEMVs on the same weights."""
import numpy as np
import pytest

from conftest import rel_l2, say
from midge_amd import DevBuf, device, synth
from midge_amd.moe import MoELayer, expert_major_dev
from midge_amd.synth import Keys, MoEShape

pytestmark = pytest.mark.gpu
# Three e2m3 terms leave at most 2^-12 of a 32-block's largest value, as a
# uniform error 2^-12 / sqrt(3) of it, and that value is ~2.2 rms of a normal
# block: 3.1e-4 of a product sum, once in gate/up and once in down.
TOL = 6.2e-4
COUNTS = [1, 0, 16, 31, 32, 33, 63, 64, 65, 129, 257]   # tokens of each expert


@pytest.mark.parametrize("hidden,ffn,plain", [(64, 64, False), (64, 192, True), (192, 320, False), (256, 128, False),
                                              (3328, 64, False), (128, 4608, False)])
def test_gemm_edges(mh, path_switch, hidden, ffn, plain):
    say(f"prefill gemm {hidden}x{ffn} plain={plain}")
    shape = MoEShape(hidden=hidden, ffn=ffn, n_experts=len(COUNTS), top_k=2, act_plain=int(plain))
    keys = Keys(21)
    ex = synth.host_layer_experts(shape, keys, 0)
    w, s, b, nw = synth.host_router(shape, keys, 0)
    lay = MoELayer.host(shape, ex, w, s, b, nw)
    rng = np.random.default_rng(hidden + ffn)
    flat = np.concatenate([np.repeat(np.arange(len(COUNTS)), COUNTS), [-1, len(COUNTS), -1]]).astype(np.int32)
    sel = rng.permutation(flat).reshape(-1, 2)   # a token may hold one expert twice: two assignments
    n = len(sel)
    wt = rng.uniform(0.5, 1.0, (n, 2)).astype(np.float32)
    xb = rng.standard_normal((n, hidden)).astype(np.float32)
    xb[3] = 0.0
    out = []
    for gemv in (False, True):
        path_switch("NO_MFMA", gemv)
        bufs = [DevBuf.from_array(a) for a in (xb, sel, wt, np.zeros_like(xb))]
        expert_major_dev(lay, n, *bufs)
        mh.sync()
        out.append(bufs[3].download(np.float32, xb.shape))
        for d in bufs:
            d.free()
    lay.release()
    got, want = out
    assert not np.array_equal(got, want)   # the matrix cores ran
    for t in range(n):
        routed = (sel[t] >= 0) & (sel[t] < len(COUNTS))
        if not routed.any():
            assert not got[t].any()
        else:
            assert rel_l2(got[t], want[t]) < TOL, (t, sel[t])


@pytest.mark.parametrize("hidden,ffn", [(64, 64), (192, 320), (256, 128)])
@pytest.mark.parametrize("shift", [4, 8, 12])
def test_table_off_16_bytes(mh, shift, hidden, ffn):
    """Expert tables on any 4-byte boundary take the matrix cores too, with the
    same result bit for bit."""
    say(f"prefill gemm {hidden}x{ffn} table off by {shift}")
    shape = MoEShape(hidden=hidden, ffn=ffn, n_experts=4, top_k=2)
    keys = Keys(22)
    ex = synth.host_layer_experts(shape, keys, 0)
    w, s, b, nw = synth.host_router(shape, keys, 0)
    n = 150
    rng = np.random.default_rng(shift)
    sel = np.argsort(rng.random((n, 4)), axis=1)[:, :2].astype(np.int32)
    wt = rng.uniform(0.5, 1.0, (n, 2)).astype(np.float32)
    xb = rng.standard_normal((n, hidden)).astype(np.float32)
    out = []
    for off in (0, shift):
        table = DevBuf.from_array(np.concatenate([np.zeros(off, np.uint8), ex.view(np.uint8).ravel()]))
        lay = MoELayer.host(shape, table.ptr + off, w, s, b, nw)
        bufs = [DevBuf.from_array(a) for a in (xb, sel, wt, np.zeros_like(xb))]
        device.profile_enable()
        device.profile_reset()
        expert_major_dev(lay, n, *bufs)
        mh.sync()
        assert device.profile_query("moe_gu_mfma")[1] == 1
        device.profile_enable(False)
        out.append(bufs[3].download(np.float32, xb.shape))
        lay.release()
        for d in bufs + [table]:
            d.free()
    assert np.array_equal(*out) and np.abs(out[0]).max() > 0
