"""Elementwise values that several clusters read: evaluated in each of them instead of
stored, and clusters that share operands emitted as one kernel with several outputs.
Every op still rounds to its dtype, so the results equal a numpy restatement of the
graph op by op (bf16: rounded after every op) bit for bit where the ops are exact in
fp32 (products, sums), whatever the plan."""
import numpy as np
import pytest

from gomlx_hip import synth
from gomlx_hip.backend import Backend, dtypes, make_shape

pytestmark = pytest.mark.gpu

F32, BF16 = dtypes.Float32, dtypes.BFloat16


@pytest.fixture(scope="module")
def be(cuda):
    b = Backend("")
    yield b
    b.Finalize()


def _run(be, build, inputs):
    b = be.Builder("copies")
    f = b.Main()
    p = [f.Parameter(f"p{i}", s) for i, (_, s) in enumerate(inputs)]
    f.Return(build(f, *p))
    ex = b.Compile()
    plan = ex.Plan()
    outs = ex.Execute([be.BufferFromFlatData(0, a, s) for a, s in inputs])
    res = [be.BufferToFlatData(y).reshape(be.BufferShape(y).dims).copy() for y in outs]
    ex.Finalize()
    return res, plan


# 65536 elements is where clusters start to share a kernel; odd counts have a tail.
@pytest.mark.parametrize("shape", [(7, 33), (256, 256), (641, 257), (64, 8192)])
@pytest.mark.parametrize("dt", [F32, BF16])
def test_shared_values(be, shape, dt):
    rnd = synth.round_bf16 if dt == BF16 else (lambda v: np.asarray(v, np.float32))
    feed = synth.to_bf16_bits if dt == BF16 else (lambda v: v)
    back = synth.bf16_bits_to_f32 if dt == BF16 else (lambda v: v)
    x, y, z, row = (rnd(synth.normal(9100 + i, s)) for i, s in enumerate([shape, shape, shape, shape[-1:]]))
    S = make_shape(dt, *shape)

    def build(f, x, y, z, row):
        rb = f.BroadcastInDim(row, S, [1])
        d = f.Sub(x, rb)              # three readers, one large operand: evaluated in each
        q = f.Mul(d, d)               # read with d: goes along
        a = f.Add(f.Mul(d, y), q)     # a and b share x, y: one kernel where large enough
        b = f.Sub(f.Mul(q, y), d)
        m = f.Mul(f.Add(y, z), d)     # y + z has two large operands and two readers: stored
        n = f.Sub(f.Add(y, z), q)
        s = f.ReduceMax(f.Mul(d, z), 1)
        return [a, b, m, n, s]

    got, plan = _run(be, build, [(feed(v), s) for v, s in
                                 zip((x, y, z, row), (S, S, S, make_shape(dt, shape[-1])))])
    d = rnd(x - row)
    q = rnd(d * d)
    yz = rnd(y + z)
    want = [rnd(rnd(d * y) + q), rnd(rnd(q * y) - d), rnd(yz * d), rnd(yz - q), rnd(d * z).max(1)]
    for g, w in zip(got, want):
        assert np.array_equal(back(g), w), plan
    assert ("outputs=" in plan) == (shape[0] * shape[1] >= 65536), plan


def test_value_with_other_readers_is_stored_once(be):
    """A copied value's operand that is a graph output, or a product, is not recomputed."""
    S = make_shape(BF16, 128, 512)
    W = make_shape(BF16, 512, 512)
    x, w, y = synth.normal(9201, (128, 512)), synth.normal(9202, (512, 512), std=0.05), synth.normal(9203, (128, 512))

    def build(f, x, w, y):
        g = f.DotGeneral(x, [1], [], w, [0], [])
        s = f.Mul(g, y)
        return [s, f.Add(s, y), f.Mul(f.Neg(s), x), f.Sub(f.Neg(s), y)]

    got, plan = _run(be, build, [(synth.to_bf16_bits(x), S), (synth.to_bf16_bits(w), W), (synth.to_bf16_bits(y), S)])
    g = [synth.bf16_bits_to_f32(v) for v in got]
    xb, yb = synth.round_bf16(x), synth.round_bf16(y)
    assert plan.count("M=128 N=512 K=512") == 1, plan
    assert np.array_equal(g[1], synth.round_bf16(g[0] + yb))
    assert np.array_equal(g[2], synth.round_bf16(-g[0] * xb)) and np.array_equal(g[3], synth.round_bf16(-g[0] - yb))
