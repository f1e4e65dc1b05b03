"""The attention kernels at the edges of their tiles: query-row blocks of 16
to 64, key counts off the multiples of 4, 8 and 16, the element counts a
thread holds (64, 128, 256, 320 keys), both head dimensions, the longest rows of
each and the first past them, an unaligned qkv, and infinities beside padding."""
import math

import numpy as np
import pytest

from conftest import assert_bitexact

pytestmark = pytest.mark.gpu


def _ref(qkv, heads, dh):
    from qppocr_amd import nets
    from oracle import nets as onets
    b, t = qkv.shape[:2]
    g = nets.Graph(qkv.shape)
    g.outputs = [g.attention(0, heads, dh, 1.0 / math.sqrt(dh))]
    return onets.run_graph(g, qkv)[0].reshape(b, t, heads * dh)


@pytest.mark.parametrize("b,t,heads,dh", [
    (1, 1, 8, 32), (2, 3, 2, 32), (2, 7, 8, 32), (3, 8, 1, 32), (2, 15, 8, 32), (2, 17, 8, 32),
    (50, 61, 8, 32), (2, 65, 8, 32), (2, 127, 8, 32), (40, 129, 8, 32), (2, 136, 8, 32),
    (33, 160, 8, 32), (1, 255, 8, 32), (1, 256, 3, 32), (2, 30, 4, 64), (40, 70, 8, 64),
    (1, 171, 2, 64), (1, 179, 2, 64)])
def test_attention_tiles(gpu, oracle, b, t, heads, dh):
    from qppocr_amd import ops
    rng = np.random.default_rng(1000 * t + dh)
    qkv = rng.standard_normal((b, t, 3 * heads * dh)).astype(np.float32)
    print(f"attention {b} x {t}, {heads} x {dh}", flush=True)
    y = ops.attention(gpu.from_numpy(qkv).cuda(), heads, dh, 1.0 / math.sqrt(dh))
    assert_bitexact(y.cpu().numpy(), _ref(qkv, heads, dh), f"attention T={t}")


def test_attention_unaligned(gpu, oracle):
    """qkv four bytes past a 16-byte boundary."""
    from qppocr_amd import ops
    b, t, heads, dh = 2, 77, 8, 32
    rng = np.random.default_rng(9)
    qkv = rng.standard_normal((b, t, 3 * heads * dh)).astype(np.float32)
    buf = gpu.empty(qkv.size + 1, device="cuda")
    view = buf[1:].view(qkv.shape)
    view.copy_(gpu.from_numpy(qkv))
    assert view.data_ptr() % 16 == 4
    y = ops.attention(view, heads, dh, 1.0 / math.sqrt(dh))
    assert_bitexact(y.cpu().numpy(), _ref(qkv, heads, dh), "attention, unaligned")


def test_attention_infinite_keys(gpu, oracle):
    """An infinite query or key spoils its own rows as in the reference, and no
    padding column's 0 * inf reaches a result."""
    from qppocr_amd import ops
    b, t, heads, dh = 2, 13, 2, 32
    rng = np.random.default_rng(11)
    qkv = rng.standard_normal((b, t, 3 * heads * dh)).astype(np.float32)
    qkv[0, 4, 7] = np.inf             # a query of head 0
    qkv[1, 12, heads * dh + 40] = np.nan   # a key of head 1
    y = ops.attention(gpu.from_numpy(qkv).cuda(), heads, dh, 1.0 / math.sqrt(dh)).cpu().numpy()
    ref = _ref(qkv, heads, dh)
    assert_bitexact(y[0, [0, 1, 2, 3, 5, 12]], ref[0, [0, 1, 2, 3, 5, 12]], "rows beside inf")
    assert_bitexact(y[1, :, :32], ref[1, :, :32], "head beside NaN")
    assert np.isfinite(y[0, :, 32:]).all()


def test_attention_past_lds(gpu):
    """Head dimension 64 takes 179 keys; the general kernel has no room for more."""
    from qppocr_amd import ops
    from qppocr_amd._lib import QphError
    qkv = gpu.zeros((1, 180, 3 * 2 * 64), device="cuda")
    with pytest.raises(QphError, match="too large for LDS"):
        ops.attention(qkv, 2, 64, 0.125)


def _plan_attention(qkv, heads, dh, scale):
    """The seven dispatches of a planned attention (one launch when run)."""
    from test_gpu_plan import MiniPlan
    b, t = qkv.shape[:2]
    part, bh = b * heads * t * dh, b * heads
    mp = MiniPlan()
    x, sc = mp.static(qkv), mp.static(np.array([scale, 0, 0, 0], np.float32))
    t5, qs, kt = mp.alloc(3 * part), mp.alloc(part), mp.alloc(part)
    s, p = mp.alloc(bh * t * t), mp.alloc(bh * t * t)
    o, y = mp.alloc(part), mp.alloc(part)
    mp.dispatch("n_transpose_nd", [x, t5, 3 * part, 5, b, t, 3, heads, dh, 2, 0, 3, 1, 4])
    mp.dispatch("n_elem", [7, t5, sc, qs, part, 0.0, 0.0])
    mp.dispatch("n_transpose_nd", [t5 + part, kt, part, 4, b, heads, t, dh, 0, 0, 1, 3, 2, 0])
    mp.dispatch("n_attn_mm", [qs, kt, s, t, dh, t, bh, heads], (1, bh * t, 1))
    mp.dispatch("n_softmax", [s, p, bh * t, t, t, heads * t], (bh * t, 1, 1))
    mp.dispatch("n_attn_mm", [p, t5 + 2 * part, o, t, t, dh, bh, heads], (1, bh * t, 1))
    mp.dispatch("n_transpose_nd", [o, y, part, 4, b, heads, t, dh, 0, 0, 2, 1, 3, 0])
    mp.output(y, part, (b, t, heads * dh))
    return mp


@pytest.mark.parametrize("b,t,heads", [(1, 257, 2), (3, 304, 1), (1, 311, 2), (9, 312, 8)])
def test_plan_attention_long_rows(gpu, oracle, b, t, heads):
    """Rows past 256 keys, which only a plan holds: 320 elements a row's eight threads."""
    rng = np.random.default_rng(t)
    qkv = rng.standard_normal((b, t, 3 * heads * 32)).astype(np.float32)
    scale = 1.0 / math.sqrt(32)
    print(f"plan attention {b} x {t}, {heads} x 32", flush=True)
    got = _plan_attention(qkv, heads, 32, scale).run()[0]
    assert_bitexact(got, _ref(qkv, heads, 32), f"plan attention T={t}")


def test_plan_attention_past_lds(gpu):
    from qppocr_amd._lib import QphError
    with pytest.raises(QphError, match="too large for LDS"):
        _plan_attention(np.zeros((1, 313, 96), np.float32), 1, 32, 0.125).run()
