"""ppocr_rh_probs_dev recorded in a HIP graph and replayed on other inputs.  A replay runs the
recorded launches under the epochs they were recorded with, so each of its passes must find
the precision guard's list empty.  The inputs of two replays in a row guard more than half of
the rows each, and other rows, so rows left from the replay before would push new ones out of
the list, and would take the three-term statistics without the three-term probabilities.  Every
replay is compared with the eager call on the same inputs, bit for bit; the program works on
the GPU between the replays."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

RELAXED = 2  # hipStreamCaptureModeRelaxed


class _Graph:
    """The launches of `call` on a stream, recorded once."""

    def __init__(self, stream, call):
        from ppocr_rechead.hip import check, hip
        g = ctypes.c_void_p()
        self.exec = ctypes.c_void_p()
        check(hip().hipStreamBeginCapture(stream.h, RELAXED), "hipStreamBeginCapture")
        try:
            call()
        finally:
            rc = hip().hipStreamEndCapture(stream.h, ctypes.byref(g))
        check(rc, "hipStreamEndCapture")
        check(hip().hipGraphInstantiate(ctypes.byref(self.exec), g, None, None, ctypes.c_size_t(0)), "hipGraphInstantiate")
        check(hip().hipGraphDestroy(g), "hipGraphDestroy")
        self.stream = stream

    def replay(self):
        from ppocr_rechead.hip import check, hip
        check(hip().hipGraphLaunch(self.exec, self.stream.h), "hipGraphLaunch")
        self.stream.synchronize()

    def close(self):
        from ppocr_rechead.hip import check, hip
        check(hip().hipGraphExecDestroy(self.exec), "hipGraphExecDestroy")


# label, FP32 head, mode, m, n, outlier weights, rows' scale where they are guarded
CASES = [
    # a grid of more than two workgroups per CU: a rescue launch over the row list
    ("row list", False, 2, 6000, 4001, False, 30.0),
    # outlier weights lower the limit below 4: whole row blocks are listed by the scan and skipped
    ("skipped blocks", False, 2, 1500, 1000, True, 1.0),
    # in-kernel rescue of the statistics; the writer alone lists rows
    ("small batch", False, 2, 300, 500, False, 30.0),
    # guarded rows of an FP32 head, recomputed in fp32 products
    ("fp32 rescue", True, 3, 1500, 1000, False, 60.0),
]


@pytest.mark.parametrize("label,fp32,mode,m,n,outliers,big", CASES, ids=[c[0] for c in CASES])
def test_replayed_probabilities_equal_the_eager_call(rh, label, fp32, mode, m, n, outliers, big):
    from ppocr_rechead.hip import H2D, DeviceArray, Stream, check, hip, synchronize
    rng = np.random.default_rng(m + n)
    w = (rng.standard_normal((n, 120)) * 0.05).astype(np.float32)
    if outliers:
        w[rng.choice(n, n // 50, replace=False), rng.integers(0, 120)] = 5.0
    bias = (rng.standard_normal(n) * 0.01).astype(np.float32)
    head = rh.RecHead(w_t=w, bias=bias) if fp32 else rh.RecHead(qw=rh.QuantizedWeight.from_f32_transposed(w), bias=bias)
    inputs = []
    for lo, hi in ((0, 3 * m // 5), (2 * m // 5, m), (0, 0), (m // 5, 4 * m // 5)):
        a = (rng.standard_normal((m, 120)) * (0.1 if outliers else 1.0)).astype(np.float32)
        a[lo:hi] = rng.standard_normal((hi - lo, 120)).astype(np.float32) * np.float32(big)
        g = head.guarded_rows(a, mode)
        assert (g[lo:hi].all() and hi - lo > m // 2) or hi == lo, label
        assert not np.delete(g, np.s_[lo:hi]).any(), label
        inputs.append(a)
    print(f"graph replay: {label}, {m} rows, {n} classes, limits {head.guard_limits(mode)}", flush=True)
    L, st = rh._lib.lib(), Stream()
    ws = head.workspace_bytes(m, mode)
    da, dout, dws = DeviceArray((m, 120), np.float32), DeviceArray((m, n), np.float32), DeviceArray((ws,), np.uint8)
    eager_out, eager_ws = DeviceArray((m, n), np.float32), DeviceArray((ws,), np.uint8)
    dws.fill_bytes(0)
    eager_ws.fill_bytes(0)

    def put(a):
        check(hip().hipMemcpy(da.p, a.ctypes.data_as(ctypes.c_void_p), ctypes.c_size_t(a.nbytes), H2D), "hipMemcpy H2D")

    def call(out, work):
        rh._check(L.ppocr_rh_probs_dev(head.handle, da.p, m, mode, out.p, work.p, ws, st.h))

    put(inputs[0])
    call(dout, dws)  # code objects are loaded before the capture
    st.synchronize()
    graph = _Graph(st, lambda: call(dout, dws))
    for turn, which in enumerate((0, 1, 3, 0, 2, 1, 1)):
        put(inputs[which])
        graph.replay()
        got = dout.numpy()
        call(eager_out, eager_ws)
        synchronize()
        want = eager_out.numpy()
        bad = np.nonzero((got.view(np.uint32) != want.view(np.uint32)).any(axis=1))[0]
        assert bad.size == 0, f"{label}: replay {turn} differs in {bad.size} rows, first {bad[:5]}"
    graph.close()
    head.close()
    for d in (da, dout, dws, eager_out, eager_ws):
        d.free()
