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
    (9000, 192, 1010, "gelu"), (9000, 256, 1000, "res"),
    (1700, 320, 530, "gelu"), (4300, 320, 250, "res"), (5300, 1024, 250, "plain"),  # rounds 4 to 6
    (2700, 320, 513, "plain")])
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


@pytest.mark.parametrize("n,c,m", [(1, 64, 8), (1, 256, 1280), (2, 256, 1280), (33, 1280, 64),
                                   (3, 64, 6), (2, 96, 32), (1, 1024, 204)])
def test_session_single_pixel_conv(gpu, oracle, n, c, m):
    """1x1 convs of single-pixel maps over the batch, with the bias rules of one
    item (seeded from 2e5 products on) and of several, and the shapes that stay
    a GEMM per item (M % 4, C % 64)."""
    from qppocr_amd import _lib, nets
    from oracle import nets as onets
    rng = np.random.default_rng(n * c + m)
    g = nets.Graph((n, c, 1, 1))
    w = g.weight((rng.standard_normal((m, c, 1, 1)) / np.sqrt(c)).astype(np.float32))
    b = g.weight(rng.standard_normal(m).astype(np.float32))
    g.outputs = [g.conv(0, w, b, act=_lib.ACT_HARDSWISH)]
    x = rng.standard_normal((n, c, 1, 1)).astype(np.float32)
    print(f"1x1 conv {n} x {c} -> {m}", flush=True)
    sess = nets.HipSession(g)
    for k in {n, 1}:      # every item, and one with the rest padding
        got = sess.run(x[:k])[0]
        g1 = nets.Graph((k, c, 1, 1))
        g1.weights = g.weights
        g1.outputs = [g1.conv(0, w, b, act=_lib.ACT_HARDSWISH)]
        assert_bitexact(got, onets.run_graph(g1, x[:k])[0], f"1x1 conv {k} of {n}")
    sess.close()


@pytest.mark.parametrize("rows", [1280, 1159, 1153, 577])
def test_session_wide_linear_rows(gpu, oracle, rows):
    """The one-wave GEMM's row stores with a partial last row block."""
    from qppocr_amd import nets
    from oracle import nets as onets
    rng = np.random.default_rng(rows)
    k, n = 32, 18709 if rows == 577 else 9001
    g = nets.Graph((rows, 1, 1, k))
    w = g.weight((rng.standard_normal((k, n)) / np.sqrt(k)).astype(np.float32))
    logits = g.linear(0, w, g.weight(rng.standard_normal(n).astype(np.float32)))
    g.outputs = list(g.softmax_argmax(logits, n))
    x = rng.standard_normal((rows, 1, 1, k)).astype(np.float32)
    print(f"wide linear {rows} x {k} x {n}", flush=True)
    sess = nets.HipSession(g)
    got = sess.run(x)
    sess.close()
    ref = onets.run_graph(g, x)
    assert_bitexact(got[0], ref[0], f"probabilities {rows}x{n}")
    assert (np.ascontiguousarray(got[1]).view(np.uint32) ==
            np.ascontiguousarray(ref[1]).view(np.uint32)).all()


@pytest.mark.parametrize("rows,n,form", [(1280, 9001, "relu"), (1159, 9001, "res"), (1280, 9001, "plain"),
                                         (1280, 9024, "relu")])
def test_session_wide_linear_softmax(gpu, oracle, rows, n, form):
    """A linear of the wide size between an activation or a residual and the
    softmax that alone reads it: its rows may lie padded, 32 floats apart."""
    from qppocr_amd import _lib, nets
    from oracle import nets as onets
    rng = np.random.default_rng(rows + n)
    k = 64
    w = (rng.standard_normal((k, n)) / np.sqrt(k)).astype(np.float32)
    b = (rng.standard_normal(n) * 0.1).astype(np.float32)
    g = nets.Graph((rows, 1, 1, k))
    res = -1
    if form == "res":
        w0 = (rng.standard_normal((k, n)) / np.sqrt(k)).astype(np.float32)
        res = g.linear(0, g.weight(w0), g.weight(b[::-1].copy()), act=_lib.ACT_RELU)
    y = g.linear(0, g.weight(w), g.weight(b), residual=res,
                 act=_lib.ACT_RELU if form == "relu" else _lib.ACT_NONE)
    g.outputs = list(g.softmax_argmax(y, n))
    x = rng.standard_normal((rows, 1, 1, k)).astype(np.float32)
    print(f"wide linear + softmax {rows} x {k} x {n} {form}", flush=True)
    sess = nets.HipSession(g)
    got = sess.run(x)
    sess.close()
    ref = onets.run_graph(g, x)
    assert_bitexact(got[0], ref[0], f"probabilities {rows}x{n} {form}")
    assert (np.ascontiguousarray(got[1]).view(np.uint32) ==
            np.ascontiguousarray(ref[1]).view(np.uint32)).all()
