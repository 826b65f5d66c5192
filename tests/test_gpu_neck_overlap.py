"""The tail with its output over its inputs' memory: d_out as d_x, as d_shortcut, and shifted
against either where that is allowed (a shortcut of token rows only as the same buffer).  The
bits of the same call on separate buffers, at the row counts of every tile size of the block
kernels and of the separate kernels, with two blocks and with one (whose first kernel is also
the last to read x)."""
import numpy as np
import pytest

from neck_common import DIM, neck_weights, rows_to_cf
from test_gpu_neck import _inputs, _make

pytestmark = pytest.mark.gpu

# lines that lie across the tiles of rows; 16400: the separate kernels
LENGTHS = {120: [120], 333: [120, 90, 3, 120], 4096: [120] * 34 + [16], 8100: [270] * 30, 16384: [512] * 32,
           16400: [400] * 41}


@pytest.mark.parametrize("blocks", [1, 2])
@pytest.mark.parametrize("m", sorted(LENGTHS))
@pytest.mark.parametrize("cf", [False, True], ids=["rows", "channels first"])
def test_output_over_the_inputs(rh, cf, m, blocks):
    from ppocr_rechead.hip import DeviceArray, synchronize
    w = neck_weights(seed=61, blocks=blocks)
    neck = _make(rh, w)
    x, sc, off = _inputs(LENGTHS[m], seed=22)
    assert x.shape[0] == m
    if cf:
        x, sc = rows_to_cf(x, off), rows_to_cf(sc, off)
    layout = rh.NECK_CHANNELS_FIRST if cf else rh.NECK_ROWS
    wsb = neck.workspace_bytes(m)
    doff, dws = DeviceArray.from_numpy(off), DeviceArray((wsb,), np.uint8)
    size = m * DIM

    def run(label, out_on, shift):
        """The call with out starting `shift` floats from the start of x ("x"), of the
        shortcut ("shortcut"), or in memory of its own."""
        print(f"tail overlap: {label}, {m} rows, {blocks} blocks, channels first {cf}", flush=True)
        at = max(0, -shift)  # floats before the input in its buffer
        bufs = {}
        for name, v in (("x", x), ("shortcut", sc)):
            b = np.zeros(size + abs(shift), np.float32)
            b[at:at + size] = v.reshape(-1)
            bufs[name] = DeviceArray.from_numpy(b)
        own = DeviceArray((size,), np.float32)
        ptr = {k: v.p.value + 4 * at for k, v in bufs.items()}
        dst = ptr[out_on] + 4 * shift if out_on else own.p.value
        rh._check(rh._lib.lib().ppocr_rn_forward_dev(neck.handle, ptr["x"], ptr["shortcut"], m, doff.p, len(off) - 1,
                                                     layout, dst, dws.p, wsb, None))
        synchronize()
        got = bufs[out_on].numpy()[at + shift:at + shift + size] if out_on else own.numpy()
        for b in (*bufs.values(), own):
            b.free()
        return got

    want = run("separate", None, 0)
    step = 64 * DIM if m > 200 else 8 * DIM
    calls = [("x", 0), ("x", step), ("x", -step), ("shortcut", 0)]
    if cf:
        calls += [("shortcut", step), ("shortcut", -step)]
    for out_on, shift in calls:
        got = run(f"out on {out_on} {shift:+d}", out_on, shift)
        assert np.array_equal(got, want), (out_on, shift)
    neck.close()
    for d in (doff, dws):
        d.free()
