"""Depthwise + pointwise blocks in the register-fed kernel: tiles of 16, 32 and
64 pixels, rows that are no multiple of four pixels (unaligned loads, chunks
past a row's and the image's ends, partial groups), single-group rows, slices of M past eight channel blocks, several
images, and the channel-last store."""
import numpy as np
import pytest

from conftest import assert_bitexact

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,c,m,h,w,k,s,trans", [
    (1, 16, 32, 7, 3, 3, 1, False), (1, 32, 32, 9, 26, 3, 1, False),
    (1, 32, 32, 130, 270, 3, 1, False), (1, 16, 32, 200, 416, 3, 2, False),
    (2, 32, 64, 33, 53, 3, 2, False), (1, 64, 64, 61, 130, 3, 1, False),
    (1, 64, 64, 192, 192, 3, 1, False), (3, 64, 128, 13, 13, 3, 2, False),
    (1, 128, 128, 10, 26, 3, 1, False), (1, 128, 128, 5, 13, 5, 1, False),
    (1, 128, 128, 96, 96, 5, 1, False), (1, 128, 256, 11, 27, 3, 2, False),
    (1, 128, 130, 4, 1, 3, 1, False), (2, 128, 17, 3, 5, 5, 1, False),
    (1, 32, 48, 1, 2, 3, 1, False), (9, 64, 64, 12, 48, 3, 1, False),
    (2, 32, 64, 6, 21, 3, 2, True),
    (1, 16, 16, 1, 1, 5, 1, False), (2, 16, 32, 1, 1, 3, 2, False), (1, 16, 16, 9, 1, 5, 1, False),
    (3, 16, 16, 2, 3, 5, 1, False), (1, 16, 16, 1, 7, 3, 1, False), (2, 32, 32, 2, 2, 3, 2, False),
    (1, 64, 64, 17, 18, 5, 1, False), (2, 128, 128, 17, 19, 3, 2, False),
    (1, 128, 128, 16, 18, 5, 1, False), (2, 16, 16, 31, 405, 3, 2, False)])
def test_dwpw_tiles(gpu, oracle, n, c, m, h, w, k, s, trans):
    from qppocr_amd import _lib, nets
    from oracle import nets as onets
    rng = np.random.default_rng(c * 1000 + h * w + m)
    g = nets.Graph((n, c, h, w))
    f32 = lambda a: np.asarray(a, np.float32)  # noqa: E731
    wd = g.weight(f32(rng.standard_normal((c, 1, k, k)) / k))
    bd = g.weight(f32(rng.standard_normal(c) * 0.1))
    wp = g.weight(f32(rng.standard_normal((m, c, 1, 1)) / np.sqrt(c)))
    bp = g.weight(f32(rng.standard_normal(m) * 0.1))
    t = g.conv(0, wd, bd, stride=(s, s), pad=(k // 2,) * 4, group=c, act=_lib.ACT_HARDSWISH)
    y = g.conv(t, wp, bp, act=_lib.ACT_RELU if m == 48 else _lib.ACT_HARDSWISH, trans_out=trans)
    g.outputs = [y]
    x = rng.standard_normal((n, c, h, w)).astype(np.float32)
    print(f"dw {k}x{k} s{s} + pw {n}x{c}x{h}x{w} -> {m}", flush=True)
    sess = nets.HipSession(g)
    assert sess.plan()[0][1] == 2      # one launch of both nodes
    got = sess.run(x)[0]
    sess.close()
    assert_bitexact(got, onets.run_graph(g, x)[0], f"dw+pw {n}x{c}x{h}x{w} -> {m}")
