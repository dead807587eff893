"""The long-matrix batched int8 kernel (k_gemm_q8r_rows) against the register-
operand kernel on the same digits: their int32 sums are exact, so every output
is the same bit for bit. Sizes at the edges of its column groups (16-column
tiles, up to 4), K steps (one chunk of 64, odd and even counts, rows of whole
4 KB, whose steps go round from a start of each block's own) and row tiles (a
partial last tile, rows not a multiple of 4)."""
import numpy as np
import pytest

from conftest import say
from midge_amd import DT_Q8R, DevBuf
from midge_amd.kern import WT, matvec_dev

pytestmark = pytest.mark.gpu
LONG = 131072   # rows from which the long tiling fills a 256-CU card


@pytest.mark.parametrize("rows,cols,batch", [(LONG, 64, 2), (LONG + 5, 192, 17), (LONG + 20, 128, 33), (LONG + 3, 640, 64),
                                             (LONG + 48, 320, 65), (LONG + 16, 64, 130), (201088, 2880, 16),
                                             (LONG, 4096, 3), (LONG + 37, 8192, 20)])
def test_rows_kernel_bit_identical(mh, path_switch, rows, cols, batch):
    say(f"q8 rows kernel {rows}x{cols} batch={batch}")
    rng = np.random.default_rng(rows + batch)
    W = rng.integers(-127, 128, (rows, cols), dtype=np.int8)
    sc = rng.uniform(1e-3, 1e-2, rows).astype(np.float32)
    X = rng.standard_normal((batch, cols)).astype(np.float32)
    X[0] = 0.0
    if rows == LONG:
        X[1, 7] = np.inf   # a column that takes the plain f32 sum
    bufs = [DevBuf.from_array(a) for a in (W, sc, X)]
    yd = DevBuf(4 * batch * rows)
    t = WT(DT_Q8R, rows, cols, bufs[0].ptr, bufs[1].ptr)
    out = []
    for other in (False, True):
        path_switch("Q8_NO_ROWS", other)
        matvec_dev(t, bufs[2], yd, batch)
        out.append(yd.download(np.float32, (batch, rows)))
    for d in bufs + [yd]:
        d.free()
    assert np.array_equal(out[0], out[1], equal_nan=True)
    assert not out[0][0].any()
    r = rng.choice(rows, 64, replace=False)
    r[0] = rows - 1
    fin = np.isfinite(X).all(1)
    want = (X[fin].astype(np.float64) @ W[r].T.astype(np.float64)) * sc[r]
    # x held to 2^-22 of its largest value, sums exact
    bound = np.abs(X[fin]).max(1)[:, None] * 2.0 ** -22 * np.abs(W[r]).sum(1) * sc[r] + 2.0 ** -22 * np.abs(want)
    assert (np.abs(out[0][fin][:, r] - want) <= bound).all()
