"""The block kernels of the tail (neck_fused.hip) where they can go wrong: lines around the
16-row query blocks and the 64-key steps, tiles that hold many lines, empty lines, more lines
than the 512 of one window of the line table, the row counts where the tile grows (4096 and
8192 rows) and where the separate kernels take over (16384).  Lines are independent, so the
oracle runs some lines of each batch; the bar is the tail's (tests/test_gpu_neck.py)."""
import ctypes

import numpy as np
import pytest

from neck_common import DIM, neck_weights, oracle_neck, rows_to_cf
from test_gpu_neck import _check, _inputs, _make

pytestmark = pytest.mark.gpu


def _many(seed, lines, hi):
    return np.random.default_rng(seed).integers(0, hi + 1, lines).tolist()


CASES = [
    ("around the tiles", [15, 1, 16, 17, 63, 64, 65, 0, 128, 129, 31, 33]),
    ("one row each", [1] * 45),
    ("windows of the line table", _many(1, 1500, 3)),
    ("lines at the windows' edges", [2] * 511 + [0, 0, 5, 1] + [1] * 700),
    ("tiles of 16, last one whole", [64] * 64),
    ("tiles of 32", [64] * 64 + [1]),
    ("tiles of 64", [8193 - 120 * 68] + [120] * 68),
    ("separate kernels", [120] * 136 + [65]),
    ("a long line", [700, 3]),
]


@pytest.mark.parametrize("label,lengths", CASES, ids=[c[0] for c in CASES])
def test_block_kernels_at_their_edges(orc, rh, label, lengths):
    w = neck_weights(seed=51)
    neck = _make(rh, w)
    x, sc, off = _inputs(lengths, seed=19)
    print(f"neck blocks: {label}, {int(off[-1])} rows, {len(lengths)} lines", flush=True)
    got = neck.forward(x, sc, off)
    full = [b for b in range(len(lengths)) if lengths[b] > 0]
    for b in sorted({full[0], full[1], full[len(full) // 2], full[-2], full[-1]}):
        t0, t1 = int(off[b]), int(off[b + 1])
        ref = oracle_neck(orc, w, x[t0:t1], sc[t0:t1], np.array([0, t1 - t0]))
        _check(got[t0:t1], ref, f"{label}: line {b}")
    got_cf = neck.forward(rows_to_cf(x, off), rows_to_cf(sc, off), off, layout=rh.NECK_CHANNELS_FIRST)
    assert np.array_equal(got_cf, got)
    neck.close()


def test_a_line_of_nan_stays_alone(rh):
    """Lines share tiles of rows; a NaN in one reaches none of the others' outputs."""
    w = neck_weights(seed=52)
    neck = _make(rh, w)
    x, sc, off = _inputs([20, 7, 50], seed=20)
    want = neck.forward(x, sc, off)
    x[off[1] + 2, 5] = np.nan
    got = neck.forward(x, sc, off)
    assert np.isnan(got[off[1]:off[2]]).any()
    assert np.array_equal(got[:off[1]], want[:off[1]]) and np.array_equal(got[off[2]:], want[off[2]:])
    neck.close()


def test_unaligned_input_rows(rh):
    """Input rows 4 bytes off a 16-byte boundary: the same bits as the aligned ones."""
    from ppocr_rechead.hip import DeviceArray, synchronize
    w = neck_weights(seed=53)
    neck = _make(rh, w)
    x, sc, off = _inputs([33, 90], seed=21)
    m = int(off[-1])
    want = neck.forward(x, sc, off)
    dx = DeviceArray.from_numpy(np.concatenate([[0.0], x.reshape(-1)]).astype(np.float32))
    ds, doff, dout = DeviceArray.from_numpy(sc), DeviceArray.from_numpy(off), DeviceArray((m, DIM), np.float32)
    wsb = neck.workspace_bytes(m)
    dws = DeviceArray((wsb,), np.uint8)
    rh._check(rh._lib.lib().ppocr_rn_forward_dev(neck.handle, ctypes.c_void_p(dx.p.value + 4), ds.p, m, doff.p, 2,
                                                 rh.NECK_ROWS, dout.p, dws.p, wsb, None))
    synchronize()
    assert np.array_equal(dout.numpy(), want)
    for d in (dx, ds, doff, dout, dws):
        d.free()
    neck.close()


@pytest.mark.parametrize("lengths", [[33, 90], [120] * 40, [240] * 40], ids=["tiles of 16", "tiles of 32", "tiles of 64"])
@pytest.mark.parametrize("cf", [False, True], ids=["rows", "channels first"])
def test_unaligned_rows(rh, cf, lengths):
    """Each of x, the shortcut and the output, and all of them, 4 bytes off a 16-byte boundary:
    the same bits as the aligned ones, and nothing written around the output."""
    from ppocr_rechead.hip import DeviceArray, synchronize
    w = neck_weights(seed=53)
    neck = _make(rh, w)
    x, sc, off = _inputs(lengths, seed=21)
    m = int(off[-1])
    want = neck.forward(x, sc, off)
    if cf:
        x, sc = rows_to_cf(x, off), rows_to_cf(sc, off)
    doff = DeviceArray.from_numpy(off)
    wsb = neck.workspace_bytes(m)
    dws = DeviceArray((wsb,), np.uint8)
    for mask in (1, 2, 4, 7):
        at = [1 if mask >> b & 1 else 0 for b in range(3)]
        ds = [DeviceArray.from_numpy(np.concatenate([np.zeros(o), v.reshape(-1), np.zeros(4)]).astype(np.float32))
              for o, v in zip(at, (x, sc))]
        dout = DeviceArray.from_numpy(np.full(m * DIM + 5, 7.0, np.float32))
        ptr = [ctypes.c_void_p(d.p.value + 4 * o) for d, o in zip((*ds, dout), at)]
        rh._check(rh._lib.lib().ppocr_rn_forward_dev(neck.handle, ptr[0], ptr[1], m, doff.p, len(lengths),
                                                     rh.NECK_CHANNELS_FIRST if cf else rh.NECK_ROWS, ptr[2], dws.p, wsb,
                                                     None))
        synchronize()
        got = dout.numpy()
        assert np.array_equal(got[at[2]:at[2] + m * DIM].reshape(m, DIM), want), mask
        assert np.all(got[:at[2]] == 7.0) and np.all(got[at[2] + m * DIM:] == 7.0), mask
        for d in (*ds, dout):
            d.free()
    for d in (doff, dws):
        d.free()
    neck.close()
