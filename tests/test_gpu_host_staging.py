"""Host decode calls whose inputs end around the staging pieces (512 KB), leave the stage (4 MB),
and whose results leave the pinned buffer (256 KB): the bits of one device call."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_host_decode_across_the_staging_sizes(rh, orc):
    from ppocr_rechead.hip import DeviceArray, synchronize
    rng = np.random.default_rng(5)
    w = (rng.standard_normal((200, 120)) * 0.05).astype(np.float32)
    q, s = orc.pack_int8(w)
    head = rh.RecHead(qw=rh.QuantizedWeight(q, s), bias=np.zeros(200, np.float32))
    L = rh._lib.lib()
    for m in (1, 1092, 1093, 2184, 2185, 8737, 8738, 24000, 1092):
        a = rng.standard_normal((m, 120)).astype(np.float32)
        off = np.array([0, m // 3, m], np.int64)
        got = head.decode(a, off, 2)
        da, doff = DeviceArray.from_numpy(a), DeviceArray.from_numpy(off)
        di, dm, dq = DeviceArray((m,), np.int32), DeviceArray((m,), np.float32), DeviceArray((m,), np.int32)
        dl, ds = DeviceArray((2,), np.int64), DeviceArray((2,), np.float32)
        ws = head.workspace_bytes(m, 2)
        dw = DeviceArray((ws,), np.uint8)
        rh._check(L.ppocr_rh_decode_dev(head.handle, da.p, m, doff.p, 2, 2, di.p, dm.p, dq.p, dl.p, ds.p, dw.p, ws, None))
        synchronize()
        assert np.array_equal(got["idx"], di.numpy()), m
        assert np.array_equal(got["maxprob"], dm.numpy()), m
        assert np.array_equal(got["score"], ds.numpy()), m
        sl, sq = dl.numpy(), dq.numpy()
        for b in range(2):
            assert np.array_equal(got["seqs"][b], sq[off[b]:off[b] + sl[b]]), (m, b)
        for d in (da, doff, di, dm, dq, dl, ds, dw):
            d.free()
    head.close()


def test_host_decode_nct_across_the_staging_sizes(rh, orc):
    """The same for the channels-first entry, whose one input and results are staged alike."""
    from ppocr_rechead.hip import DeviceArray, synchronize
    rng = np.random.default_rng(6)
    w = (rng.standard_normal((200, 120)) * 0.05).astype(np.float32)
    q, s = orc.pack_int8(w)
    head = rh.RecHead(qw=rh.QuantizedWeight(q, s), bias=np.zeros(200, np.float32))
    L = rh._lib.lib()
    for lines, steps in ((1, 1), (4, 273), (3, 364), (8, 273), (19, 115), (79, 110), (24, 365), (200, 120), (4, 273)):
        m = lines * steps
        x = rng.standard_normal((lines, 120, steps)).astype(np.float32)
        got = head.decode_nct(x, 2)
        dx = DeviceArray.from_numpy(x)
        di, dm, dq = DeviceArray((m,), np.int32), DeviceArray((m,), np.float32), DeviceArray((m,), np.int32)
        dl, ds = DeviceArray((lines,), np.int64), DeviceArray((lines,), np.float32)
        ws = head.workspace_bytes(m, 2)
        dw = DeviceArray((ws,), np.uint8)
        rh._check(L.ppocr_rh_decode_nct_dev(head.handle, dx.p, lines, steps, 2, di.p, dm.p, dq.p, dl.p, ds.p, dw.p, ws, None))
        synchronize()
        assert np.array_equal(got["idx"], di.numpy()), m
        assert np.array_equal(got["maxprob"], dm.numpy()), m
        assert np.array_equal(got["score"], ds.numpy()), m
        sl, sq = dl.numpy(), dq.numpy()
        for b in range(lines):
            assert np.array_equal(got["seqs"][b], sq[b * steps:b * steps + sl[b]]), (m, b)
        for d in (dx, di, dm, dq, dl, ds, dw):
            d.free()
    head.close()


def test_host_argmax_and_ctc_across_the_pinned_results(rh):
    """ppocr_argmax_rows and ppocr_ctc_greedy with results around 256 KB, where they leave the
    pinned buffer."""
    rng = np.random.default_rng(7)
    for rows in (1, 32767, 32768, 32769):  # two results of 128 KB
        x = rng.standard_normal((rows, 5)).astype(np.float32)
        idx, val = np.zeros(rows, np.int32), np.zeros(rows, np.float32)
        rh._check(rh._lib.lib().ppocr_argmax_rows(rh._ptr(x), rows, 5, rh._ptr(idx), rh._ptr(val)))
        assert np.array_equal(idx, x.argmax(axis=1)) and np.array_equal(val, x.max(axis=1)), rows
    for steps in (1, 64, 65000, 65400, 65536, 65600):  # the tokens, 8 + 4 bytes a line
        ids = rng.integers(0, 3, steps).astype(np.int32)
        p = rng.random(steps).astype(np.float32)
        off = np.array([0, steps // 3, steps], np.int64)
        seqs, score = rh.CtcDecoder.collapse(ids, p, off)
        for b in range(2):
            i = ids[off[b]:off[b + 1]]
            keep = i != 0
            keep[1:] &= i[1:] != i[:-1]
            assert np.array_equal(seqs[b], i[keep]), (steps, b)
            total = np.float32(0.0)
            for v in p[off[b]:off[b + 1]][keep]:
                total += v
            assert score[b] == (total / np.float32(keep.sum()) if keep.any() else 0.0), (steps, b)
