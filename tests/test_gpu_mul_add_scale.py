"""mul_add_scale over small planes (four elements a thread across plane
borders), around its 1024-element limit and on planes that are not whole
quads.  Bit-exact against the oracle."""
import numpy as np
import pytest

from conftest import assert_bitexact

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,c,h,w", [(1, 1, 1, 4), (3, 7, 6, 6), (2, 256, 3, 12), (1, 5, 31, 33),
                                     (1, 3, 30, 34), (1, 3, 32, 32), (2, 3, 5, 5), (1, 300, 2, 2)])
def test_mul_add_scale_small_planes(gpu, oracle, n, c, h, w):
    import torch
    from qppocr_amd import ops
    r = np.random.default_rng(n + c * h + w)
    x, res = (r.standard_normal((n, c, h, w)).astype(np.float32) for _ in range(2))
    gate = r.standard_normal((1, c, 1, 1)).astype(np.float32)
    print(f"mul_add_scale {n}x{c}x{h}x{w}", flush=True)
    got = ops.mul_add_scale(*(torch.from_numpy(a).cuda() for a in (x, gate, res)))
    assert_bitexact(got.cpu().numpy(), oracle.mul_add_scale(x, gate, res), "mul_add_scale")
