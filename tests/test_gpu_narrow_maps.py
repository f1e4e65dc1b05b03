"""Convs of maps whose rows are not 16-byte aligned or whole: the pointwise
kernel's one-word slab loads (1 to 512 output channels) and the LDS 3x3
kernel's one-word halo loads, the 3x3 kernel of large maps with 17 to 24
outputs, and det nets that take all of them (grouped laterals and smoothing
convs, the head's conv-transpose pair).  Bit-exact against the oracle."""
import numpy as np
import pytest

from conftest import assert_bitexact

pytestmark = pytest.mark.gpu


def _conv(gpu, oracle, n, c, h, w, m, k, res):
    import torch
    from qppocr_amd import ops
    rng = np.random.default_rng(n * c + h * w + m)
    x = rng.standard_normal((n, c, h, w)).astype(np.float32)
    wt = (rng.standard_normal((m, c, k, k)) / np.sqrt(c * k * k)).astype(np.float32)
    b = (rng.standard_normal(m) * 0.1).astype(np.float32)
    p = k // 2
    ref = oracle.conv2d(x, wt, b, oracle.conv_params(1, 1, p, p))
    r = rng.standard_normal(ref.shape).astype(np.float32) if res else None
    if res:
        ref = oracle.binary_flat(ref, r, 0)
    print(f"conv {k}x{k} {n}x{c}x{h}x{w} -> {m}", flush=True)
    got = ops.conv2d(*(torch.from_numpy(a).cuda() for a in (x, wt, b)), ops.conv_params(1, 1, p, p),
                     residual=torch.from_numpy(r).cuda() if res else None)
    assert_bitexact(got.cpu().numpy(), ref, "conv")


@pytest.mark.parametrize("n,c,h,w,m,res", [
    (1, 16, 1, 1, 1, False), (1, 16, 1, 15, 16, True), (2, 48, 1, 17, 17, False),
    (3, 32, 5, 13, 96, True), (1, 256, 5, 13, 96, False), (1, 64, 33, 33, 129, False),
    (2, 32, 7, 9, 300, True), (1, 32, 151, 151, 151, False),
    (1, 16, 520, 512, 40, False),     # two row blocks a wave, one past M
    (2, 128, 101, 163, 96, True), (1, 256, 129, 129, 96, False),   # two, three
    (4, 32, 128, 128, 48, True), (4, 16, 120, 113, 20, False),     # all of M in a wave
    (1, 256, 160, 160, 256, True), (4, 768, 41, 39, 120, False),   # four; three, one past M
    (1, 16, 200, 103, 512, False), (4, 128, 6, 6, 512, True)])
def test_conv1x1_any_map(gpu, oracle, n, c, h, w, m, res):
    _conv(gpu, oracle, n, c, h, w, m, 1, res)


@pytest.mark.parametrize("n,c,h,w,m,res", [
    (1, 8, 320, 1, 24, False), (1, 24, 161, 33, 32, True), (2, 96, 81, 63, 24, False),
    (5, 32, 64, 31, 5, False), (1, 40, 107, 90, 17, True),
    (1, 32, 78, 98, 32, False), (1, 32, 80, 98, 32, False),    # 156 and 160 tiles
    (1, 8, 128, 97, 16, True), (1, 24, 120, 94, 32, True), (1, 16, 107, 90, 17, False),
    (4, 96, 64, 98, 24, False), (1, 40, 270, 95, 20, True), (4, 8, 120, 113, 9, False)])
def test_conv3x3_any_width(gpu, oracle, n, c, h, w, m, res):
    _conv(gpu, oracle, n, c, h, w, m, 3, res)


@pytest.mark.parametrize("n,c,h,w,m,res", [
    (1, 8, 481, 97, 24, True), (1, 16, 477, 128, 17, False),   # 484 and 480 tiles
    (3, 24, 161, 124, 23, False), (1, 40, 479, 100, 20, True), (2, 32, 240, 127, 24, False),
    (4, 8, 37, 400, 24, True)])     # 520 tiles, but 988 of two rows
def test_conv3x3_tall(gpu, oracle, n, c, h, w, m, res):
    _conv(gpu, oracle, n, c, h, w, m, 3, res)


@pytest.mark.parametrize("h,w", [(96, 160), (224, 416), (512, 544), (960, 992)])
def test_det_net_odd_coarse_levels(gpu, oracle, h, w):
    from qppocr_amd import nets
    from oracle import nets as onets
    g, x = nets.build_det(3, h, w)
    print(f"det {h}x{w}", flush=True)
    sess = nets.HipSession(g)
    got = sess.run(x)[0]
    sess.close()
    assert_bitexact(got, onets.run_graph(g, x)[0], "det map")
