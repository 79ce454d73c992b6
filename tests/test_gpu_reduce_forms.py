"""The generated reduce kernels' forms (rows, columns, general; whole or split into
ranges) at the sizes where the form, vector width or launch shape changes, against
numpy in float64, and with a fused producer bit for bit against the unfused plan.

Bounds: a sum of n fp32 terms in any order is within n 2^-24 of sum |x| (here far
fewer terms meet in one accumulator: 2^-20 is allowed); the result of a 16-bit
reduction rounds once more (2^-8 bf16, 2^-11 f16).  Maxima and integers are exact."""
import numpy as np
import pytest

from gomlx_hip import synth
from gomlx_hip.backend import Backend, dtypes, make_shape

pytestmark = pytest.mark.gpu

F32, BF16, F16, I32 = dtypes.Float32, dtypes.BFloat16, dtypes.Float16, dtypes.Int32
# (shape, reduced axes)
CASES = [
    ((3, 64), [1]), ((5, 1000), [1]), ((7, 1002), [1]), ((4, 513), [1]),          # rows, a wave each
    ((1, 10000), [1]), ((600, 4096), [1]), ((2, 3, 40, 128), [2, 3]),             # wider groups, two axes
    ((3, 1 << 20), [1]), ((256, 10), [0, 1]),                                     # split rows; everything
    ((64, 8), [0]), ((2000, 64), [0]), ((7, 50, 24), [1]), ((3, 129, 9), [1]),    # columns
    ((4096, 2048), [0]), ((2, 70000, 8), [1]), ((513, 130), [0]), ((6, 5, 4, 40), [1, 2]),
    ((6, 40, 5), [0, 2]), ((70, 3), [0]), ((9, 7, 3), [1]),                       # general, wave and thread
    ((8193, 2, 8), [1]), ((8200, 3, 24), [1]), ((70001, 5, 9), [1]), ((16384, 7, 20), [1]),  # threads, 1 to 4 wide
    ((70000, 63, 8), [1]), ((33000, 2, 3, 64), [1, 2]),
    ((0, 8), [0]), ((8, 0), [1]),                                                 # nothing to reduce
]


@pytest.fixture(scope="module")
def be(cuda):
    b = Backend("")
    yield b
    b.Finalize()


def _run(be, shape, axes, dt, op, feed, square):
    b = be.Builder("reduce")
    f = b.Main()
    x = f.Parameter("x", make_shape(dt, *shape))
    f.Return([getattr(f, op)(f.Mul(x, x) if square else x, *axes)])
    ex = b.Compile()
    buf = be.BufferFromFlatData(0, feed, make_shape(dt, *shape))
    (y,) = ex.Execute([buf])
    s = be.BufferShape(y)
    out = be.BufferToFlatData(y).reshape(s.dims).copy()
    plan = ex.Plan()
    ex.Finalize()
    return (synth.bf16_bits_to_f32(out) if dt == BF16 else out), plan


@pytest.mark.parametrize("shape,axes", CASES)
@pytest.mark.parametrize("dt", [F32, BF16, F16, I32])
def test_reduce_forms(be, shape, axes, dt, monkeypatch):
    if dt == I32:
        x = synth.uniform_f32(9001, shape, -1000, 1000).astype(np.int32)
        feed = x
    else:
        x = synth.normal(9001, shape)
        feed = synth.to_bf16_bits(x) if dt == BF16 else x.astype(np.float16) if dt == F16 else x
        x = synth.round_bf16(x) if dt == BF16 else feed.astype(np.float32)
    print(shape, axes, dt, flush=True)
    x64 = x.astype(np.float64)
    ax = tuple(axes)
    got, plan = _run(be, shape, axes, dt, "ReduceSum", feed, False)
    want = x64.sum(ax)
    if dt == I32:
        assert np.array_equal(got, want.astype(np.int64).astype(np.int32))
    else:
        err = np.abs(got.astype(np.float64) - want)
        r = {F32: 0.0, BF16: 2.0 ** -8, F16: 2.0 ** -11}[dt]
        assert np.all(err <= 2.0 ** -20 * np.abs(x64).sum(ax) + r * np.abs(want) + 2.0 ** -24), plan
    if x.size:
        assert np.array_equal(_run(be, shape, axes, dt, "ReduceMax", feed, False)[0].astype(np.float64), x64.max(ax))
    fused, plan = _run(be, shape, axes, dt, "ReduceSum", feed, True)
    monkeypatch.setenv("GHIP_REDUCE_FUSION", "0")
    plain, _ = _run(be, shape, axes, dt, "ReduceSum", feed, True)
    assert "producer fused" in plan and np.array_equal(fused, plain, equal_nan=True)


def test_grid_beyond_x(be):
    """More workgroups than a grid takes in x: they go on in y (int8; rows and columns,
    fused with their operand)."""
    for dims, axis in [((1 << 24, 64), 1), ((1 << 22, 64, 8), 1)]:
        b = be.Builder("grid")
        f = b.Main()
        S = make_shape(dtypes.Int8, *dims)
        r = f.Parameter("r", make_shape(dtypes.Int8, *dims[1:]))
        i = f.ConvertDType(f.Rem(f.Iota(make_shape(dtypes.Int32, *dims), 0), f.Constant(np.int32(101))), dtypes.Int8)
        f.Return([f.ReduceMax(f.Add(i, f.BroadcastInDim(r, S, list(range(1, len(dims))))), axis), f.ReduceMax(i, axis)])
        ex = b.Compile()
        print(dims, ex.Plan(), flush=True)
        row = (np.arange(np.prod(dims[1:])) % 13).astype(np.int8).reshape(dims[1:])
        got = ex.Execute([be.BufferFromFlatData(0, row, make_shape(dtypes.Int8, *dims[1:]))])
        base = (np.arange(dims[0]) % 101).astype(np.int8)
        tail = row.max(0)
        want = [base[:, None] + tail.reshape(1, -1), np.broadcast_to(base[:, None], (dims[0], tail.size))]
        for y, w in zip(got, want):
            assert np.array_equal(be.BufferToFlatData(y).reshape(dims[0], -1), w)
            be.BufferFinalize(y)
        ex.Finalize()


def test_split_reduce_says_so(be):
    for shape, axes in [((3, 1 << 20), [1]), ((4096, 2048), [0])]:
        b = be.Builder("reduce")
        f = b.Main()
        f.Return([f.ReduceSum(f.Parameter("x", make_shape(F32, *shape)), *axes)])
        ex = b.Compile()
        assert "ranges)" in ex.Plan()
        ex.Finalize()


VIEWS = [  # (operand shape, permutation, last-axis slice stride, reduced axes of the view)
    ((40, 96, 130), (0, 1, 2), 1, [2]), ((40, 96, 130), (2, 0, 1), 1, [2]), ((40, 96, 130), (1, 2, 0), 2, [0]),
    ((40, 96, 128), (0, 1, 2), 2, [1]), ((5, 6, 7, 72), (2, 0, 3, 1), 1, [1, 3]), ((5, 6, 7, 72), (1, 3, 0, 2), 1, [0, 2]),
    ((4, 3, 2, 5, 64), (0, 2, 1, 3, 4), 1, [2, 3]), ((9, 70, 8), (0, 1, 2), 1, [1]), ((2, 3, 4096), (1, 0, 2), 1, [1, 2]),
]


@pytest.mark.parametrize("shape,perm,stride,axes", VIEWS)
@pytest.mark.parametrize("op", ["ReduceSum", "ReduceProduct", "ReduceMax", "ReduceMin"])
@pytest.mark.parametrize("dt,npt", [(dtypes.Int8, np.int8), (dtypes.Uint8, np.uint8), (dtypes.Int16, np.int16),
                                    (dtypes.Uint16, np.uint16), (dtypes.Uint32, np.uint32), (dtypes.Int64, np.int64),
                                    (dtypes.Uint64, np.uint64), (dtypes.Float64, np.float64), (F32, np.float32)])
def test_strided_operands(be, shape, perm, stride, axes, op, dt, npt):
    """Every dtype and operation over transposed and strided views, small whole numbers:
    exact (sums and products of the integer types wrap)."""
    u = synth.uniform_f32(9101, shape, 0, 1)
    signed = np.issubdtype(npt, np.signedinteger) or npt in (np.float32, np.float64)
    if op == "ReduceProduct":  # mostly ones
        x = np.where(u < 0.03, 2, np.where((u > 0.97) & signed, -1, 1)).astype(npt)
    else:
        x = (np.floor(u * 100) - (50 if signed else 0)).astype(npt)
    print(shape, perm, stride, axes, op, dt, flush=True)
    b = be.Builder("strided")
    f = b.Main()
    v = f.Transpose(f.Parameter("x", make_shape(dt, *shape)), *perm)
    dims = [shape[p] for p in perm]
    if stride > 1:
        v = f.Slice(v, [0] * len(dims), dims, [1] * (len(dims) - 1) + [stride])
    f.Return([getattr(f, op)(v, *axes)])
    ex = b.Compile()
    (y,) = ex.Execute([be.BufferFromFlatData(0, x, make_shape(dt, *shape))])
    got = be.BufferToFlatData(y).reshape(be.BufferShape(y).dims)
    ex.Finalize()
    view = x.transpose(perm)[..., ::stride]
    fn = {"ReduceSum": np.sum, "ReduceProduct": np.prod, "ReduceMax": np.max, "ReduceMin": np.min}[op]
    want = fn(view, axis=tuple(axes), **({"dtype": npt} if op in ("ReduceSum", "ReduceProduct") else {}))
    assert np.array_equal(got, want)
