"""The plan model's windowed kernels at the sizes where they can go wrong:
the depthwise window (one or two pixels a thread, blocks of 64 or 256) on maps
smaller than the window, ragged and past the block rule, and the
conv-transpose pair (16 pixels a wave, 64 a workgroup) on maps around those
counts.  Bit-exact against the oracle."""
import pytest

from conftest import assert_bitexact
from test_gpu_plan import OFF_NONE, MiniPlan, nhwc, rnd, rng

pytestmark = pytest.mark.gpu

DW = [  # n, c, h, w, k, (sh, sw), (pt, pl, pb, pr)
    (1, 4, 1, 1, 3, (1, 1), (1, 1, 1, 1)),
    (1, 4, 1, 1, 5, (1, 1), (2, 2, 2, 2)),
    (3, 8, 2, 3, 5, (1, 1), (2, 2, 2, 2)),         # map smaller than the window, odd width
    (1, 20, 7, 9, 3, (2, 2), (1, 1, 1, 1)),
    (2, 12, 9, 11, 5, (1, 2), (2, 1, 2, 3)),       # uneven pads
    (1, 16, 12, 33, 3, (2, 1), (0, 1, 2, 1)),
    (1, 8, 130, 127, 3, (1, 1), (1, 1, 1, 1)),     # 64-thread blocks
    (1, 32, 129, 131, 3, (1, 1), (1, 1, 1, 1)),    # past 2^17 threads: 256-thread blocks
    (2, 64, 96, 97, 5, (1, 1), (2, 2, 2, 2)),      # the same, two pixels a thread
]


@pytest.mark.parametrize("case", DW, ids=lambda c: "n%d_c%d_%dx%d_k%d" % c[:5])
def test_plan_depthwise_window(gpu, oracle, case):
    from qppocr_amd import plan
    n, c, h, w, k, (sh, sw), pads = case
    r = rng(c * h + w + k)
    x, wt, b = rnd(r, (n, c, h, w)), rnd(r, (c, 1, k, k), 1.0 / k), rnd(r, (c,), 0.1)
    ref = oracle.relu_inplace(oracle.conv2d(x, wt, b, oracle.conv_params(sh, sw, *pads, group=c)).copy())
    oh, ow = ref.shape[2:]
    mp = MiniPlan()
    xo, wo = mp.static(nhwc(x)), mp.static(plan.repack_dw_w(wt, c, k, k))
    bo, yo = mp.static(plan.conv_bias(b, c)), mp.alloc(n * oh * ow * c)
    mp.dispatch("n_conv_dw", [xo, wo, bo, yo, oh * ow, c, ow, w, h, k * k, k, sh, sw, pads[0],
                              pads[1], 2, *plan.GELU_C, OFF_NONE], (1, n, 1))
    mp.output(yo, n * oh * ow * c, (n, oh, ow, c))
    print(f"plan dw window {case}", flush=True)
    assert_bitexact(mp.run()[0], nhwc(ref), "depthwise")


@pytest.mark.parametrize("n,h,w,co", [(1, 1, 1, 1), (1, 4, 4, 4), (2, 3, 5, 3), (1, 8, 8, 1),
                                      (3, 9, 13, 2)])
def test_plan_convt_pair_sizes(gpu, oracle, n, h, w, co):
    from qppocr_amd import plan
    r = rng(n + 10 * h + w + co)
    x = rnd(r, (n, 24, h, w))
    w1, w2 = rnd(r, (24, 24, 2, 2), 0.3), rnd(r, (24, co, 2, 2), 0.3)
    b1, b2 = rnd(r, (24,), 0.2), rnd(r, (co,), 0.2)
    t = oracle.convtranspose2d(x, w1) + b1[None, :, None, None]
    t = oracle.convtranspose2d(oracle.relu_inplace(t.copy()), w2) + b2[None, :, None, None]
    ref = oracle.sigmoid_tensor(t)
    mp = MiniPlan()
    xo = mp.static(nhwc(x))
    wo1 = mp.static(plan.repack_convt_w(w1, 24, 24, 2, 2))
    wo2 = mp.static(plan.repack_convt_w(w2, 24, co, 2, 2))
    bo1, bo2 = mp.static(plan.conv_bias(b1, 24)), mp.static(plan.conv_bias(b2, co))
    y1, y2 = mp.alloc(n * 4 * h * w * 24), mp.alloc(n * 16 * h * w * 4)
    mp.dispatch("n_convt", [xo, wo1, bo1, y1, 4 * h * w, 24, 2 * w, w, h, 24, 6, 2, 2, 2, 2,
                            *plan.GELU_C], (1, n, 1))
    mp.dispatch("n_convt", [y1, wo2, bo2, y2, 16 * h * w, 4, 4 * w, 2 * w, 2 * h, 24, 6, 2, 2, 2, 0,
                            *plan.GELU_C], (1, n, 1))
    out = mp.alloc(n * 16 * h * w * co)
    mp.dispatch("n_exit", [y2, out, n, co, 4 * h, 4 * w, 4, 4])
    mp.output(out, n * 16 * h * w * co, (n, co, 4 * h, 4 * w))
    mp.p.total_words = mp.words
    print(f"plan convt pair {n} {h}x{w} -> {co}", flush=True)
    s = plan.HipPlanSession(mp.p)
    try:
        assert s.launches() == 1
        (got,) = s.run(None)
    finally:
        s.close()
    assert_bitexact(got, ref, "conv-transpose pair + exit")
