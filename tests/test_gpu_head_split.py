"""The session's fused head over a split weight (two float16 terms a value):
row counts at the edges of its tiles (32 rows a wave, 64 of the small form,
256 of a workgroup), column counts that leave a partial block of 32, ties,
rows of extreme scale, and rows with an infinity or a NaN, which take the
float32 order of the unsplit kernels."""
import math

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

K = 256


def _session(rows, w, b):
    from qppocr_amd import nets
    g = nets.Graph((rows, 1, 1, K))
    logits = g.linear(0, g.weight(w), g.weight(b))
    g.outputs = [g.softmax_argmax(logits, w.shape[1], probs=False)[1]]
    g.flags |= nets.NET_FUSED_HEAD
    return nets.HipSession(g)


def _weights(n, seed):
    rng = np.random.default_rng(seed)
    w = (rng.standard_normal((K, n)) * math.sqrt(2 / K)).astype(np.float32)
    b = (rng.standard_normal(n) * 0.1).astype(np.float32)
    return rng, w, b


def _ref(x, w, b):
    z = x.astype(np.float64) @ w.astype(np.float64) + b
    z = np.sort(z, axis=1), z.argmax(1), z
    top = z[0][:, -1]
    with np.errstate(over="ignore"):
        p = 1.0 / np.exp(z[2] - top[:, None]).sum(1)
    return p, z[1], top - z[0][:, -2]


@pytest.mark.parametrize("rows,n", [(1, 18709), (31, 100), (32, 32), (33, 1001), (64, 33),
                                    (65, 18709), (255, 97), (256, 64), (257, 18709), (1100, 3001),
                                    (6800, 18709)])
def test_head_split_matches_float64(gpu, rows, n):
    rng, w, b = _weights(n, rows + n)
    x = rng.standard_normal((rows, K)).astype(np.float32) * 2
    x[0] = 0.0                         # the biases alone: a row without a scale
    b[n // 3] = b[n - 1] = 9.0         # ... with a tie, the first wins
    w[:, n // 3] = w[:, n - 1] = 0.0
    if rows > 40:
        x[7] *= 1e-6                   # rows far from the others' scale
        x[33] *= 1e3
        x[40, 1:] = 0.0
    print(f"head split {rows} x {K} x {n}", flush=True)
    sess = _session(rows, w, b)
    pairs = sess.run(x.reshape(rows, 1, 1, K))[0].reshape(rows, 2)
    sess.close()
    p, idx, gap = _ref(x, w, b)
    ids = np.ascontiguousarray(pairs[:, 1]).view(np.uint32)
    assert ids[0] == n // 3
    assert (ids[1:] == idx[1:])[gap[1:] > 1e-4].all()
    # a logit is within 60 roundings of its magnitude (48 of the accumulator,
    # the scaling, the bias); the value's relative error is its logits' error
    big = np.abs(x.astype(np.float64)) @ np.abs(w).max(1).astype(np.float64) + np.abs(b).max()
    assert (np.abs(pairs[:, 0] - p) <= p * (60 * 2.0 ** -24 * big + 1e-6)).all()


def test_head_split_closer_than_the_float32_chain(gpu):
    """Against float64, over rows and weights of the rec head's scale, the pair
    values are no further off than the unsplit kernels'."""
    torch = gpu
    from qppocr_amd import ops
    rng, w, b = _weights(18709, 3)
    x = rng.standard_normal((320, K)).astype(np.float32) * 2
    sess = _session(320, w, b)
    got = sess.run(x.reshape(320, 1, 1, K))[0].reshape(320, 2)[:, 0]
    sess.close()
    t = lambda a: torch.from_numpy(a).cuda()  # noqa: E731
    old = ops.linear_softmax_argmax(t(x), t(w), t(b)).cpu().numpy()[:, 0]
    p, _, _ = _ref(x, w, b)
    err = lambda v: np.linalg.norm(v - p) / np.linalg.norm(p)  # noqa: E731
    print("relative error, split / float32 chain:", err(got), err(old))
    assert err(got) <= err(old)


@pytest.mark.parametrize("rows", [40, 300])
def test_head_split_rows_with_infinities(gpu, rows):
    """Rows that hold an infinity, a NaN or a magnitude past 2^60 give the
    unsplit kernels' bits; the rows beside them are not touched."""
    torch = gpu
    from qppocr_amd import ops
    rng, w, b = _weights(1001, rows)
    x = rng.standard_normal((rows, K)).astype(np.float32)
    x[3, 5], x[17, 0], x[18, 255], x[rows - 1, 9] = np.inf, np.nan, -np.inf, 3e19
    sess = _session(rows, w, b)
    pairs = sess.run(x.reshape(rows, 1, 1, K))[0].reshape(rows, 2)
    clean = x.copy()
    odd = [3, 17, 18, rows - 1]
    clean[odd] = 1.0
    beside = sess.run(clean.reshape(rows, 1, 1, K))[0].reshape(rows, 2)
    sess.close()
    t = lambda a: torch.from_numpy(a).cuda()  # noqa: E731
    old = ops.linear_softmax_argmax(t(x), t(w), t(b)).cpu().numpy()
    bits = lambda a: np.ascontiguousarray(a).view(np.uint32)  # noqa: E731
    nan = np.isnan(old[odd, 0])
    assert (np.isnan(pairs[odd, 0]) == nan).all()
    assert (bits(pairs[odd, 0])[~nan] == bits(old[odd, 0])[~nan]).all()
    assert (bits(pairs[odd, 1]) == bits(old[odd, 1])).all()
    rest = np.setdiff1d(np.arange(rows), odd)
    assert (bits(pairs[rest]) == bits(beside[rest])).all()


@pytest.mark.parametrize("where", ["weight", "bias"])
def test_head_split_refuses_weights_it_cannot_hold(gpu, where):
    """An infinity among the weights keeps the session on the unsplit kernels."""
    torch = gpu
    from qppocr_amd import ops
    rng, w, b = _weights(300, 5)
    (w[7:8, 200:201] if where == "weight" else b[200:201])[...] = -np.inf
    x = np.abs(rng.standard_normal((70, K))).astype(np.float32)
    sess = _session(70, w, b)
    pairs = sess.run(x.reshape(70, 1, 1, K))[0].reshape(70, 2)
    sess.close()
    t = lambda a: torch.from_numpy(a).cuda()  # noqa: E731
    old = ops.linear_softmax_argmax(t(x), t(w), t(b)).cpu().numpy()
    assert (pairs.view(np.uint32) == old.view(np.uint32)).all()


@pytest.mark.parametrize("rows", [24, 300])
def test_head_split_distant_winner(gpu, rows):
    """A winner far above every other class, in the first blocks and in the
    last: gaps around the range of a float32 exponential and past it."""
    n, cols, gaps = 18709, [10, 40, 5000, 18708], [87.5, 88.5, 95.0, 126.0, 200.0, 3000.0]
    rng, w, b = _weights(n, rows)
    w *= 0.1
    w[:4] = 0.0
    w[range(4), cols] = 1.0             # row q of the weight moves class cols[q] alone
    x = rng.standard_normal((rows, K)).astype(np.float32)
    x[:, :4] = 0.0
    for i in range(rows):
        x[i, i % 4] = gaps[i // 4 % len(gaps)] * (-1 if i >= 4 * len(gaps) and i % 3 == 0 else 1)
    print(f"head split, distant winners, {rows} rows", flush=True)
    sess = _session(rows, w, b)
    pairs = sess.run(x.reshape(rows, 1, 1, K))[0].reshape(rows, 2)
    sess.close()
    p, idx, gap = _ref(x, w, b)
    ids = np.ascontiguousarray(pairs[:, 1]).view(np.uint32)
    assert (ids == idx)[gap > 1e-4].all()
    # logits of at most 5 beside the winner's, whose own rounding cancels: 1e-5
    # is some 40 roundings of such a logit
    assert (np.abs(pairs[:, 0] - p) <= 1e-5 * p).all()


@pytest.mark.parametrize("rows", [24, 300])
def test_head_split_logits_past_float32(gpu, rows):
    """Operands within their limit whose products are not: column 0 overflows
    a float32 sum for some rows, and is far above or below for the others."""
    rng, w, b = _weights(1001, rows)
    w[:, 0] = 1e18
    x = rng.standard_normal((rows, K)).astype(np.float32)
    x[3], x[5] = 1.1e18, -1.1e18
    x[rows - 1] = 1e12
    print(f"head split, column 0 of 1e18, {rows} rows", flush=True)
    sess = _session(rows, w, b)
    pairs = sess.run(x.reshape(rows, 1, 1, K))[0].reshape(rows, 2)
    sess.close()
    p, idx, gap = _ref(x, w, b)
    ids = np.ascontiguousarray(pairs[:, 1]).view(np.uint32)
    assert (ids == idx)[gap > 1e-4].all()
    assert (np.abs(pairs[:, 0] - p) <= 1e-5 * p).all()


@pytest.mark.parametrize("rows,terms,channel", [(64, 1, 1), (320, 4, 1), (320, 32, 1), (64, 64, 1),
                                                (320, K, 2.0 ** 23), (40, K, 2.0 ** 23)])
def test_head_split_rows_it_would_lose_on(gpu, rows, terms, channel):
    """Rows of few terms, and rows with a channel far past the others whose
    weight is 0: against float64 no further off than the unsplit kernels', whose
    logits they then have (the order of the sums apart)."""
    torch = gpu
    from qppocr_amd import ops
    rng, w, b = _weights(18709, 7)
    x = (rng.standard_normal((rows, K)) * 2 * math.sqrt(K / terms)).astype(np.float32)
    for r in x:
        r[rng.permutation(K)[terms:]] = 0.0
    if channel > 1:
        x[:, 9], w[9] = 3.0 * channel, 0.0
    print(f"head split {rows} rows of {terms} terms, channel {channel}", flush=True)
    sess = _session(rows, w, b)
    got = sess.run(x.reshape(rows, 1, 1, K))[0].reshape(rows, 2)[:, 0]
    sess.close()
    t = lambda a: torch.from_numpy(a).cuda()  # noqa: E731
    old = ops.linear_softmax_argmax(t(x), t(w), t(b)).cpu().numpy()[:, 0]
    p, _, _ = _ref(x, w, b)
    err = lambda v: np.sqrt((((v - p) / p) ** 2).mean())  # noqa: E731
    print("relative error, session / float32 chain:", err(got), err(old))
    assert err(got) <= 1.1 * err(old)


def test_head_split_refuses_columns_of_few_terms(gpu):
    torch = gpu
    from qppocr_amd import ops
    rng, w, b = _weights(300, 6)
    w[95:, 200] = 0.0
    x = rng.standard_normal((70, K)).astype(np.float32)
    sess = _session(70, w, b)
    pairs = sess.run(x.reshape(70, 1, 1, K))[0].reshape(70, 2)
    sess.close()
    t = lambda a: torch.from_numpy(a).cuda()  # noqa: E731
    old = ops.linear_softmax_argmax(t(x), t(w), t(b)).cpu().numpy()
    assert (pairs.view(np.uint32) == old.view(np.uint32)).all()
