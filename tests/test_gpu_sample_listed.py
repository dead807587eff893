"""The select launch's pick from its listed candidates (pick_listed): sizes on
both sides of the ranked and the listed way, groups of equal p inside a bin, a
bin with more candidates than are ranked (the sort decides), probabilities
over many octaves. Picks equal the oracle's."""
import numpy as np
import pytest

from conftest import say
from midge_amd import DevBuf
from midge_amd.moe import sample_dev
from oracle import pyoracle as po

pytestmark = pytest.mark.gpu


V = 60000


def logits(m, spread, ties, octaves):
    """m of V tokens above the rest: normal (groups of `ties` equal), or of p over
    `octaves` octaves with as much mass in each."""
    rng = np.random.default_rng(m + ties)
    lg = np.full(V, -60.0, np.float32)
    if octaves:
        vals = -np.log(1 + rng.random(m) * (2.0 ** octaves - 1))
    else:
        vals = np.repeat(rng.standard_normal((m + ties - 1) // ties) * spread, ties)[:m]
    lg[rng.choice(V, m, replace=False)] = vals.astype(np.float32)
    return lg


def candidates(lg, topp):
    """Tokens of the fast list, the select launch's candidates (those of the bins
    of an eighth of an octave whose mass from the top reaches topp, with its
    margin), and the octaves that those cover."""
    e = np.exp(lg - lg.max(), dtype=np.float32)
    bins = e.view(np.uint32) >> 20
    mass = np.bincount(bins, weights=e, minlength=1017)[::-1].cumsum()
    low = 1016 - int(np.argmax(mass >= topp * e.sum(dtype=np.float64) * (1 + 1e-4)))
    c = e[bins >= low]
    return int((e >= (1 - topp) / (2 * len(lg))).sum()), len(c), float(np.log2(c.max() / c.min()))


@pytest.mark.parametrize("m,spread,ties,octaves,topp,n_cand,n_oct", [
    (1200, 2.0, 1, 0, 0.5, (1, 128), 0), (1200, 2.0, 1, 0, 0.9, (129, 8192), 5), (1200, 2.0, 1, 0, 0.99, (129, 8192), 8),
    (8000, 3.0, 1, 0, 0.9, (129, 8192), 9), (8000, 3.0, 1, 0, 0.99, (129, 8192), 13), (6000, 2.0, 7, 0, 0.9, (129, 8192), 5),
    (6000, 2.0, 7, 0, 0.99, (129, 8192), 8), (3000, 0.0, 1, 0, 0.5, (129, 8192), 0), (3000, 0.0, 1, 0, 0.99, (129, 8192), 0),
    (7000, 1.0, 700, 0, 0.9, (129, 8192), 2), (5000, 0, 1, 14, 0.9, (129, 8192), 10), (5000, 0, 1, 14, 0.99, (129, 8192), 11),
    (7000, 0, 1, 20, 0.5, (1, 128), 0), (7000, 0, 1, 20, 0.9, (129, 8192), 11), (8000, 0, 1, 18, 0.99, (129, 8192), 10),
    (2000, 0, 1, 16, 0.999, (129, 8192), 11)])
def test_listed_picks(mh, m, spread, ties, octaves, topp, n_cand, n_oct):
    say(f"sample listed m={m} spread={spread} ties={ties} octaves={octaves} topp={topp}")
    lg = logits(m, spread, ties, octaves)
    fast, cand, span = candidates(lg, topp)
    assert fast > 1024 and n_cand[0] <= cand <= n_cand[1] and span >= n_oct, (fast, cand, span)   # the select launch's
    ld, out = DevBuf.from_array(lg), DevBuf(4)
    st = 0x1234567 + m
    us = [0.0, 0.9999999]
    for _ in range(6):
        u, st = po.rng_f(st)
        us.append(u)
    for u in us:
        sample_dev(ld, V, 1.0, topp, u, out)
        got, want = int(out.download(np.int32, (1,))[0]), po.sample(lg, 1.0, topp, u)
        assert got == want, (topp, u, got, want)
    ld.free()
    out.free()
