"""The attention kernels at the edges of their tiles: query-row blocks of 16
to 64, key counts off the multiples of 4, 8 and 16, the element counts a
thread holds (64, 128, 256 keys), both head dimensions, an unaligned qkv, and
infinities beside padding."""
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
    (1, 171, 2, 64)])
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
