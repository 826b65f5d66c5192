"""The fp32 MFMA kernel (PPOCR_MODE_FP32_FMA) at the edges of its tiles: rows and classes
around 128, chunks of k around 16 and their groups of 8, k that is no multiple of 4 (the
value-by-value operand path) and 64 tiles of classes, from which the writer deals tiles to
the XCDs.  Against 64 bits: k products summed in fp32 one after another, then the scale and
the bias, differ by at most (k + 2) 2^-24 sum |a| |w| + 2^-24 |bias| (each rounding at most
half an ulp of a partial sum, which never exceeds the sum of the magnitudes)."""
import numpy as np
import pytest

from gpu_common import check_argmax, top2_gap

pytestmark = pytest.mark.gpu

CASES = [  # (m, n, k)
    (1, 1, 1), (127, 129, 4), (128, 128, 8), (129, 127, 12), (33, 300, 15), (257, 640, 16), (5, 129, 20),
    (130, 257, 24), (64, 8191, 80), (129, 8193, 120), (200, 18710, 120), (31, 500, 121), (40, 260, 200),
]


@pytest.mark.parametrize("fp32", [False, True])
@pytest.mark.parametrize("m,n,k", CASES)
def test_fp32_tiles(orc, rh, m, n, k, fp32):
    rng = np.random.default_rng(m * 7 + n * 3 + k + fp32)
    w = (rng.standard_normal((n, k)) * 0.05).astype(np.float32)
    bias = (rng.standard_normal(n) * 0.01).astype(np.float32)
    a = rng.standard_normal((m, k)).astype(np.float32)
    if fp32:
        head, wd = rh.RecHead(w_t=w, bias=bias), w.astype(np.float64)
    else:
        q, s = orc.pack_int8(w)
        head = rh.RecHead(qw=rh.QuantizedWeight(q, s), bias=bias)
        wd = q.astype(np.float64) * s.astype(np.float64)[:, None]
    print(f"fp32 tiles m={m} n={n} k={k} fp32={fp32}", flush=True)
    ref = a.astype(np.float64) @ wd.T + bias.astype(np.float64)
    mag = np.abs(a).astype(np.float64) @ np.abs(wd).T + np.abs(bias)
    bound = (k + 2) * 2.0**-24 * mag
    got = head.logits(a, 0)
    assert np.all(np.abs(got - ref) <= bound), float(np.max(np.abs(got - ref) / bound))
    d = head.decode(a, np.array([0, m], np.int64), 0)
    p = head.probs(a, 0)
    head.close()
    check_argmax(d["idx"], ref.argmax(axis=1), top2_gap(ref) if n > 1 else np.full(m, np.inf), tol=2 * bound.max())
    e = np.exp(ref - ref.max(axis=1, keepdims=True))
    pr = e / e.sum(axis=1, keepdims=True)
    # logits off by d move a probability by at most 2 d of itself; exp2, the sum over n classes
    # and its inverse add a few 2^-24 each
    rel = 2 * bound.max() + 4e-6
    assert np.all(np.abs(p - pr) <= rel * pr + 1e-30)
    assert np.all(np.abs(d["maxprob"] - pr.max(axis=1)) <= rel * pr.max(axis=1))


def _chunks(head, m):
    """Vocabulary chunks of the statistics pass, from the partials' share of the workspace."""
    def up(x):
        return (x + 255) // 256 * 256
    return (head.workspace_bytes(m, 0) - 256 - 3 * up(4 * m) - up((m + 127) // 128)) // (12 * m)


@pytest.mark.parametrize("fp32", [False, True])
@pytest.mark.parametrize("k", [4, 15, 16, 20, 32, 121])
@pytest.mark.parametrize("n", [385, 1025])
def test_statistics_over_several_tiles(orc, rh, n, k, fp32):
    """So many row blocks that a workgroup walks several tiles of classes: two, or five (one
    more than the buffers of scale and bias), with one or more chunks of k each, 4 values of k
    at a time or one by one, rows or channels first.  Sampled rows against 64 bits; the two
    layouts give the same bits."""
    rng = np.random.default_rng(n + k + fp32)
    lines, steps = 550, 120
    m = lines * steps
    w = (rng.standard_normal((n, k)) * 0.3).astype(np.float32)
    bias = (rng.standard_normal(n) * 0.5).astype(np.float32)
    if fp32:
        head, wd = rh.RecHead(w_t=w, bias=bias), w.astype(np.float64)
    else:
        q, s = orc.pack_int8(w)
        head = rh.RecHead(qw=rh.QuantizedWeight(q, s), bias=bias)
        wd = q.astype(np.float64) * s.astype(np.float64)[:, None]
    tiles = (n + 127) // 128
    per_chunk = -(-tiles // _chunks(head, m))
    print(f"fp32 statistics n={n} k={k} fp32={fp32}: {per_chunk} tiles a chunk", flush=True)
    assert per_chunk >= (2 if n == 385 else 5)
    a = rng.standard_normal((m, k)).astype(np.float32)
    off = (np.arange(lines + 1) * steps).astype(np.int64)
    got = head.decode(a, off, 0)
    cf = head.decode_nct(np.ascontiguousarray(a.reshape(lines, steps, k).transpose(0, 2, 1)), 0)
    head.close()
    assert np.array_equal(cf["idx"], got["idx"]) and np.array_equal(cf["maxprob"], got["maxprob"])
    rows = np.unique(np.concatenate([rng.choice(m, 400, replace=False), np.arange(m - 90, m)]))
    ref = a[rows].astype(np.float64) @ wd.T + bias.astype(np.float64)
    bound = (k + 2) * 2.0**-24 * (np.abs(a[rows]).astype(np.float64) @ np.abs(wd).T + np.abs(bias)).max()
    check_argmax(got["idx"][rows], ref.argmax(axis=1), top2_gap(ref), tol=2 * bound)
    p = 1.0 / np.exp(ref - ref.max(axis=1, keepdims=True)).sum(axis=1)
    assert np.all(np.abs(got["maxprob"][rows] - p) <= (2 * bound + 4e-6) * p)
