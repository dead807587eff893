"""The routers of several tokens: which one a call takes (k_combine_route,
k_route_tokens or three launches) and that its choice, weights and outputs are
those of the three launches, over the token counts, widths and expert counts at
the edges of their rules and tiles."""
import numpy as np
import pytest

from conftest import rel_l2, say
from midge_amd import DevBuf, device, synth
from midge_amd.moe import MoELayer, Stack, moe_prefill_dev
from midge_amd.synth import Keys, MoEShape

pytestmark = pytest.mark.gpu


def make(hidden, experts, top_k=2, seed=31, **kw):
    shape = MoEShape(hidden=hidden, ffn=64, n_experts=experts, top_k=top_k, **kw)
    keys = Keys(seed)
    return shape, keys, MoELayer.host(shape, synth.host_layer_experts(shape, keys, 0), *synth.host_router(shape, keys, 0))


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
