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


@pytest.mark.parametrize("m,spread,ties", [(1200, 2.0, 1), (8000, 3.0, 1), (8000, 12.0, 1), (6000, 2.0, 7), (3000, 0.0, 1),
                                           (7000, 1.0, 700)])
def test_listed_picks(mh, m, spread, ties):
    say(f"sample listed m={m} spread={spread} ties={ties}")
    rng = np.random.default_rng(m + ties)
    V = 60000
    lg = np.full(V, -60.0, np.float32)
    vals = np.repeat(rng.standard_normal((m + ties - 1) // ties) * spread, ties)[:m]
    lg[rng.choice(V, m, replace=False)] = vals.astype(np.float32)
    ld, out = DevBuf.from_array(lg), DevBuf(4)
    st = 0x1234567 + m
    for topp in (0.5, 0.9, 0.99):
        us = [0.0, 0.9999999]
        for _ in range(4):
            u, st = po.rng_f(st)
            us.append(u)
        for u in us:
            sample_dev(ld, V, 1.0, topp, u, out)
            got, want = int(out.download(np.int32, (1,))[0]), po.sample(lg, 1.0, topp, u)
            assert got == want, (topp, u, got, want)
    ld.free()
    out.free()
