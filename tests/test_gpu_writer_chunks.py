"""The logits and probabilities writer where its vocabulary chunks and its stores change: one
row, a last row block of one row (rows past the batch are dropped by the store's bounds, and
what follows the output stays as it was), the row-block counts at which the chunk count
switches, a last tile of one class, and a head of a few tiles (fewer than the chunks).
Against 64 bits: the two-term split's error stays within 5e-5 of the logits for rows inside
the guard's limit and the three-term rescue's within 1e-5, so 1e-4, the parity bar."""
import numpy as np
import pytest

from gpu_common import f64_logits_q
from test_gpu_random_shapes import _head

pytestmark = pytest.mark.gpu

CASES = [(1, 18710), (129, 18710), (500, 33), (641, 1), (2177, 2049), (2689, 2049), (4097, 4001), (9089, 257),
         (16513, 65), (33025, 97),
         # whole row blocks, with whole tiles alone and with a last tile of some classes
         (128, 64), (256, 33), (2304, 2080)]


@pytest.mark.parametrize("m,n", CASES)
def test_writer_rows_and_chunks(orc, rh, m, n):
    from ppocr_rechead.hip import DeviceArray, synchronize
    rng = np.random.default_rng(m + n)
    q, s, bias = _head(orc, rng, n, 120)
    a = rng.standard_normal((m, 120)).astype(np.float32)
    a[rng.choice(m, max(1, m // 50), replace=False)] *= np.float32(30.0)  # guarded rows
    print(f"writer m={m} n={n}", flush=True)
    head = rh.RecHead(qw=rh.QuantizedWeight(q, s), bias=bias)
    L = rh._lib.lib()
    da = DeviceArray.from_numpy(a)
    tail = 4096  # floats after the output
    dout = DeviceArray.from_numpy(np.full(m * n + tail, 7.0, np.float32))
    ws = head.workspace_bytes(m, 2)
    dws = DeviceArray((ws,), np.uint8)
    lg = f64_logits_q(a, q, s, bias)
    scale = np.maximum(1.0, np.abs(a).max(axis=1) / 4.0)[:, None]
    rh._check(L.ppocr_rh_logits_dev(head.handle, da.p, m, 2, dout.p, dws.p, ws, None))
    synchronize()
    got = dout.numpy()
    assert np.all(got[m * n:] == 7.0)
    assert np.all(np.abs(got[:m * n].reshape(m, n) - lg) <= 1e-4 * scale)
    rh._check(L.ppocr_rh_probs_dev(head.handle, da.p, m, 2, dout.p, dws.p, ws, None))
    rh._check(L.ppocr_rh_probs_dev(head.handle, da.p, m, 2, dout.p, dws.p, ws, None))  # the list emptied before each
    synchronize()
    got = dout.numpy()
    head.close()
    assert np.all(got[m * n:] == 7.0)
    e = np.exp(lg - lg.max(axis=1, keepdims=True))
    pr = e / e.sum(axis=1, keepdims=True)
    assert np.all(np.abs(got[:m * n].reshape(m, n) - pr) <= 2e-4 * scale * pr + 1e-30)
    for d in (da, dout, dws):
        d.free()


# 24 chunks in several rounds, 2 chunks, 8 chunks of more than a round of one
@pytest.mark.parametrize("m,n", [(2305, 6177), (8321, 2049), (33025, 3400)])
def test_writer_rows_sampled_from_larger_batches(orc, rh, m, n):
    """Rows from every part of the batch, among them the last row block's, in every class."""
    rng = np.random.default_rng(m + n)
    q, s, bias = _head(orc, rng, n, 120)
    a = rng.standard_normal((m, 120)).astype(np.float32)
    print(f"writer sampled m={m} n={n}", flush=True)
    head = rh.RecHead(qw=rh.QuantizedWeight(q, s), bias=bias)
    rows = np.unique(np.concatenate([rng.choice(m, 300, replace=False), np.arange(m - 130, m)]))
    got = head.logits(a, 2)[rows]
    head.close()
    scale = np.maximum(1.0, np.abs(a[rows]).max(axis=1) / 4.0)[:, None]
    assert np.all(np.abs(got - f64_logits_q(a[rows], q, s, bias)) <= 1e-4 * scale)
