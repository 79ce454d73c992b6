"""Scatters of whole rows along axis 0 through the atomic row kernel (updates that the
sorted path does not take: broadcast over scatter axes, more than 16384 rows, max / min,
integers), the sorted path's fold of a row named many times, and the fill of a broadcast
scalar, against numpy.  Integers and maxima exact; fp32 sums of k terms in any order
within k 2^-24 of sum |x|."""
import numpy as np
import pytest
import torch

from gomlx_hip import ops, synth
from gomlx_hip.backend import Backend, dtypes, make_shape

pytestmark = pytest.mark.gpu

F32, BF16, I32 = dtypes.Float32, dtypes.BFloat16, dtypes.Int32


@pytest.fixture(scope="module")
def be(cuda):
    b = Backend("")
    yield b
    b.Finalize()


def _scatter(be, mode, dt, table, ids, upd, bcast):
    """table [V, D] (op) upd rows at ids [B, L]; bcast: upd [B, D] serves all L ids."""
    V, D = table.shape
    B, L = ids.shape
    b = be.Builder("scatter")
    f = b.Main()
    p = [f.Parameter("t", make_shape(dt, V, D)), f.Parameter("i", make_shape(I32, B, L)),
         f.Parameter("u", make_shape(dt, *upd.shape))]
    u = f.BroadcastInDim(p[2], make_shape(dt, B, L, D), [0, 2]) if bcast else p[2]
    f.Return([getattr(f, mode)(p[0], f.Reshape(p[1], B, L, 1), u, 2, [2], [0], [0])])
    ex = b.Compile()
    feed = synth.to_bf16_bits if dt == BF16 else (lambda v: v)
    bufs = [be.BufferFromFlatData(0, feed(table), make_shape(dt, V, D)), be.BufferFromFlatData(0, ids, make_shape(I32, B, L)),
            be.BufferFromFlatData(0, feed(upd), make_shape(dt, *upd.shape))]
    (y,) = ex.Execute(bufs)
    out = be.BufferToFlatData(y).reshape(V, D).copy()
    plan = ex.Plan()
    ex.Finalize()
    return (synth.bf16_bits_to_f32(out) if dt == BF16 else out), plan


# D around the lane counts a row (4, 16, 64 lanes; four elements a lane)
@pytest.mark.parametrize("D", [1, 3, 7, 8, 31, 32, 255, 256, 300])
@pytest.mark.parametrize("mode", ["ScatterSum", "ScatterMax"])
@pytest.mark.parametrize("dt", [F32, BF16, I32])
def test_broadcast_rows(be, D, mode, dt):
    B, L, V = 37, 5, 50
    ids = synth.uniform_int(9401, (B, L), -2, V + 2)  # some out of range: skipped
    if dt == I32:
        table = synth.uniform_int(9402, (V, D), -1000, 1000)
        upd = synth.uniform_int(9403, (B, D), -1000, 1000)
    else:
        rnd = synth.round_bf16 if dt == BF16 else (lambda v: v)
        table, upd = rnd(synth.normal(9402, (V, D))), rnd(synth.normal(9403, (B, D)))
    got, plan = _scatter(be, mode, dt, table, ids, upd, True)
    want = table.astype(np.float64)
    mag = np.abs(want)
    fn = np.add if mode == "ScatterSum" else np.maximum
    for i in range(B):
        for k in ids[i]:
            if 0 <= k < V:
                want[k] = fn(want[k], upd[i])
                mag[k] += np.abs(upd[i])
    assert "scatter_rows_sum" not in plan
    if dt == I32 or mode == "ScatterMax":
        assert np.array_equal(got.astype(np.float64), want)
    else:
        tol = 64 * 2.0 ** -24 * mag + (2.0 ** -8 * np.abs(want) if dt == BF16 else 0)
        assert np.all(np.abs(got - want) <= tol)


def test_many_rows_and_hot_rows(be):
    """20000 rows (atomics) and 12000 rows (sorted), a third of them naming row 3."""
    V, D = 1000, 64
    for n in (20000, 12000):
        ids = synth.uniform_int(9501, (n, 1), 0, V)
        ids[::3] = 3
        upd = synth.uniform_int(9502, (n, 1, D), -8, 8).astype(np.float32)  # sums exact in fp32
        table = synth.uniform_int(9503, (V, D), -8, 8).astype(np.float32)
        got, plan = _scatter(be, "ScatterSum", F32, table, ids, upd, False)
        want = table.copy()
        np.add.at(want, ids[:, 0], upd[:, 0])
        assert ("scatter_rows_sum" in plan) == (n <= 16384)
        assert np.array_equal(got, want)


@pytest.mark.parametrize("dt", [torch.uint8, torch.bfloat16, torch.float32, torch.int64])
@pytest.mark.parametrize("n", [16, 4096, 65552, 1000003])
def test_fill(cuda, dt, n):
    src = torch.tensor([5], device=cuda).to(dt)
    out = torch.zeros(n + 16, device=cuda, dtype=dt)
    ops.copy(src.expand(n), out[:n])
    assert torch.all(out[:n] == src) and torch.all(out[n:] == 0)


# Widths around the columns a workgroup takes (64, 128, 256) and row counts around the
# rows a wave and a workgroup take, above the 4096 rows from which indices are combined.
@pytest.mark.parametrize("D", [32, 63, 64, 65, 128, 129, 257])
@pytest.mark.parametrize("rows", [4096, 4097, 4160, 5000])
@pytest.mark.parametrize("mode", ["ScatterSum", "ScatterMax"])
@pytest.mark.parametrize("dt,npt", [(F32, np.float32), (dtypes.Float64, np.float64), (I32, np.int32)])
def test_combined_rows(be, D, rows, mode, dt, npt):
    """Whole numbers, so sums are exact in any order; most rows name a few indices."""
    V = 40
    ids = np.minimum(synth.uniform_int(9501, (rows, 1), -2, V + 2), synth.uniform_int(9502, (rows, 1), -2, V + 2))
    table = synth.uniform_int(9503, (V, D), -50, 50).astype(npt)
    upd = synth.uniform_int(9504, (rows, 1, D), -50, 50).astype(npt)
    print(D, rows, mode, dt, flush=True)
    got, _ = _scatter(be, mode, dt, table, ids, upd, False)
    want, ok = table.copy(), (ids[:, 0] >= 0) & (ids[:, 0] < V)
    (np.add if mode == "ScatterSum" else np.maximum).at(want, ids[ok, 0], upd[ok, 0])
    assert np.array_equal(got, want)
