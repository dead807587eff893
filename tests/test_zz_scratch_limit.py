"""MoE calls of several tokens at the memory cap (MIDGE_HIP_MAX_BYTES): with
just the scratch that the per-assignment path needs, and at every amount above
it, a call runs and gives the uncapped result. What the faster paths take
beside it (the table of groups, the one-launch router's counters) they do
without, and a table kept by an earlier call gives way. In a child process,
which shuts the library down between the calls (fresh scratch)."""
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu
HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.mark.parametrize("kind", ["prefill", "moe", "experts"])
def test_scratch_limit(kind):
    print(f"[case] scratch limit {kind}", flush=True)
    r = subprocess.run([sys.executable, "-u", os.path.abspath(__file__), kind], capture_output=True, text=True,
                       timeout=110)
    print(r.stdout[-3000:], r.stderr[-3000:])
    assert r.returncode == 0 and "scratch limit ok" in r.stdout


def slot(nbytes):
    return max(4096, nbytes + nbytes // 4 if nbytes >= 4096 else 0)


def main(kind):
    for p in (os.path.dirname(HERE), HERE):
        if p not in sys.path:
            sys.path.insert(0, p)
    import numpy as np

    import midge_amd
    from conftest import rel_l2
    from midge_amd import DT_F32, DT_MXFP4, DT_Q4G32, DevBuf, synth
    from midge_amd.kern import WT
    from midge_amd.moe import MoELayer, expert_major_dev, moe_dev, moe_prefill_dev
    from midge_amd.synth import Keys, MoEShape

    h = f = 64
    E, k = 16, 2

    def call(dt, n, spare, before=0):
        """One call under a cap of the plain path's scratch and `spare` bytes (None: no cap), after one of `before`
        tokens with no cap."""
        midge_amd.init(0)
        shape = MoEShape(hidden=h, ffn=f, n_experts=E, top_k=k, expert_dt=dt)
        keys = Keys(3)
        ex = synth.host_layer_experts(shape, keys, 0)
        w, s, b, nw = synth.host_router(shape, keys, 0)
        wf = (w.astype(np.float32) * s[:, None]).astype(np.float32)   # an f32 router: its GEMV takes no scratch
        bufs, used = [], 0

        def dev(a):
            nonlocal used
            a = np.ascontiguousarray(a)
            bufs.append(DevBuf.from_array(a))
            used += a.nbytes
            return bufs[-1]

        x = synth.host_x(shape, keys, n, step=1)
        lay = MoELayer(shape, dev(ex).ptr, WT(DT_F32, E, h, dev(wf).ptr, 0), dev(b).ptr, dev(nw).ptr)
        sel = (np.arange(n * k, dtype=np.int32) * 5 % E).reshape(n, k)
        wt = np.full((n, k), 0.5, np.float32)
        xd, xbd, sd, wd = dev(x), dev(x), dev(sel), dev(wt)

        def go(m):
            if kind == "prefill":
                moe_prefill_dev(lay, xd, m, sd, wd)
            elif kind == "moe":
                moe_dev(lay, xd, m, sd, wd)
            else:
                expert_major_dev(lay, m, xbd, sd, wd, xd)

        if before:
            go(before)
            midge_amd.sync()
            xd.upload(x)
            sd.upload(sel)
            wd.upload(wt)
        if spare is not None:
            need = [4 * n * h, 4 * n * E, 4 * n * k * f, 4 * n * k * h, 4 * n * k, 4 * n * k]
            if n <= 16:
                need.append(8 * n * k)   # the order of a decode's GEMVs
            os.environ["MIDGE_HIP_MAX_BYTES"] = str(used + sum(slot(v) for v in need) + spare)
        try:
            go(n)
            midge_amd.sync()
        finally:
            os.environ.pop("MIDGE_HIP_MAX_BYTES", None)
        out = xd.download(np.float32, x.shape)
        for d in bufs:
            d.free()
        midge_amd.shutdown()
        return out

    for dt in (DT_MXFP4, DT_Q4G32):
        for n in (3, 40):
            want = call(dt, n, None)
            for spare in range(0, 12 * 1024 + 1, 1024):
                print(f"[case] {kind} dt {dt} n={n} spare {spare}", flush=True)
                got = call(dt, n, spare)
                assert rel_l2(got, want) < 2e-6, (n, spare, rel_l2(got, want))
    print(f"[case] {kind} after a call that kept its extras", flush=True)
    got = call(DT_MXFP4, 56, 0, before=20)
    assert rel_l2(got, call(DT_MXFP4, 56, None)) < 2e-6
    print("scratch limit ok", flush=True)
    return 0


if __name__ == "__main__":
    sys.exit(main(sys.argv[1]))
