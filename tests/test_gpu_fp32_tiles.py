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
