"""The session linears at the sizes where their tile changes (32 x 32 or 32 x 64,
two or three stages), with row and column remainders, and linears of the
one-wave GEMM's size that keep their transposed weight (activation or
residual)."""
import numpy as np
import pytest

from conftest import assert_bitexact

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,k,n,form", [
    (1280, 256, 600, "plain"),      # 760 tiles: three stages
    (1281, 192, 609, "plain"),      # 41 x 20 tiles of 32 x 32: two stages, 32 x 64
    (777, 256, 1024, "gelu"), (800, 320, 992, "res"), (2600, 192, 511, "plain"),
    (3001, 256, 300, "res"), (6200, 128, 130, "plain"),
    (9000, 192, 1010, "gelu"), (9000, 256, 1000, "res")])
def test_session_linear_tiles(gpu, oracle, rows, k, n, form):
    from qppocr_amd import _lib, nets
    from oracle import nets as onets
    rng = np.random.default_rng(rows + n)
    w = (rng.standard_normal((k, n)) / np.sqrt(k)).astype(np.float32)
    b = (rng.standard_normal(n) * 0.1).astype(np.float32)
    g = nets.Graph((rows, 1, 1, k))
    res = -1
    if form == "res":   # a residual of the output's shape: another linear's
        w0 = (rng.standard_normal((k, n)) / np.sqrt(k)).astype(np.float32)
        res = g.linear(0, g.weight(w0), g.weight(b[::-1].copy()))
    y = g.linear(0, g.weight(w), g.weight(b), residual=res,
                 act=_lib.ACT_GELU if form == "gelu" else _lib.ACT_NONE)
    g.outputs = [y]
    x = rng.standard_normal((rows, 1, 1, k)).astype(np.float32)
    print(f"linear {rows} x {k} x {n} {form}", flush=True)
    sess = nets.HipSession(g)
    got = sess.run(x)[0]
    sess.close()
    assert_bitexact(got, onets.run_graph(g, x)[0], f"linear {rows}x{k}x{n} {form}")
