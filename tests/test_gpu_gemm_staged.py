"""The register-staged GEMM cores: operands at any element alignment (odd rows,
columns, strides and bases) and grids of few tiles, against the fp64 oracle on the
same input bytes at the GEMM tolerances (fp32 results of at most a few hundred
products: 1e-4 relative to the result's RMS; one rounding to a 16-bit output), and
a fused epilogue on such operands against the unfused plan, bit for bit."""
import os

import numpy as np
import pytest
import torch

from oracle import oracle as orc
from gomlx_hip import ops, synth
from gomlx_hip.backend import ActivationType, Backend, dtypes, make_shape
from conftest import rel_err

pytestmark = pytest.mark.gpu

BF16, F16, F32 = torch.bfloat16, torch.float16, torch.float32

# (batch, M, N, K): one element, tile edges (63, 64, 65), a k-tile and one step more
# or less (32 and 64 deep), fewer columns than a 16-byte chunk, a contraction of one
# chunk, several edge tiles; and a grid of 128 x 128 tiles.
SHAPES = [(1, 1, 1, 1), (1, 63, 65, 31), (2, 65, 63, 33), (1, 64, 10, 512), (1, 256, 512, 10), (1, 10, 3, 257),
          (3, 1, 129, 63), (1, 129, 1, 65), (1, 100, 7, 129), (1, 31, 33, 1531), (1, 2049, 2055, 67),
          (700, 5, 7, 9), (700, 33, 31, 33), (300, 17, 19, 65), (150, 101, 67, 65)]  # tiles by M, N and the batch


def _operand(r, c, off, trans, dt, seed, cuda):
    """[B, r, c] values whose rows (or columns, when trans) start `off` elements into a
    wider buffer."""
    B, r, c = r[0], r[1], c
    x = synth.normal_device(seed, (B, c if trans else r, (r if trans else c) + off), std=0.125, device=cuda, dtype=dt)
    x = x[:, :, off:]
    return x.transpose(1, 2) if trans else x


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("a_t,b_t", [(False, False), (False, True), (True, False), (True, True)])
@pytest.mark.parametrize("dt,odt", [(BF16, F32), (F16, F16), (F32, F32), (F32, BF16)])
@pytest.mark.parametrize("off", [0, 3])
def test_odd_operands(cuda, shape, a_t, b_t, dt, odt, off):
    B, M, N, K = shape
    print(f"staged gemm {shape} a_t={a_t} b_t={b_t} {dt}->{odt} off={off}", flush=True)
    a = _operand((B, M), K, off, a_t, dt, 7001 + M, cuda)
    b = _operand((B, K), N, off, b_t, dt, 7101 + N, cuda)
    c = ops.gemm(a, b, out_dtype=odt).float().cpu().numpy()
    rows = np.arange(M) if M <= 300 else np.array([0, 63, 64, 127, 128, 1000, 2047, 2048])
    an = np.ascontiguousarray(a.float().cpu().numpy()[:, rows])
    ref = orc.dot_general(an, [2], [0], np.ascontiguousarray(b.float().cpu().numpy()), [1], [0])
    tol = {F32: 1e-4, F16: 1e-3, BF16: 1e-2}[odt]
    assert rel_err(c[:, rows], ref) <= tol


# fp32 grids around the 32 x 32 (contraction over the waves), 64 x 64 and 128 x 128 tiles.
@pytest.mark.parametrize("shape", [(1, 31, 33, 7), (1, 33, 31, 9), (1, 32, 32, 32), (2, 64, 96, 264), (1, 512, 1024, 40),
                                   (1, 513, 1025, 41), (1, 1536, 2048, 36), (1, 1537, 2049, 33)])
@pytest.mark.parametrize("a_t,b_t", [(False, False), (False, True), (True, False), (True, True)])
def test_f32_tile_sizes(cuda, shape, a_t, b_t):
    B, M, N, K = shape
    a = _operand((B, M), K, 0, a_t, F32, 7401, cuda)
    b = _operand((B, K), N, 0, b_t, F32, 7402, cuda)
    rows = np.unique(np.clip(np.array([0, 1, 31, 32, 33, 63, 64, 100, 511, 512, M - 2, M - 1]), 0, M - 1))
    c = ops.gemm(a, b).cpu().numpy()[:, rows]
    ref = orc.dot_general(np.ascontiguousarray(a.cpu().numpy()[:, rows]), [2], [0], np.ascontiguousarray(b.cpu().numpy()),
                          [1], [0])
    assert rel_err(c, ref) <= 1e-5


def test_values_past_the_edges_do_not_leak(cuda):
    """Neighbouring rows / columns of NaN around every odd operand stay out."""
    for dt in (BF16, F32):
        wa = torch.full((70, 80), float("nan"), device=cuda, dtype=dt)
        wb = torch.full((80, 70), float("nan"), device=cuda, dtype=dt)
        wa[1:68, 1:68] = synth.normal_device(7201, (67, 67), std=0.125, device=cuda, dtype=dt)
        wb[1:68, 1:66] = synth.normal_device(7202, (67, 65), std=0.125, device=cuda, dtype=dt)
        for a in (wa[1:68, 1:68], wa[1:68, 1:68].t().contiguous().t()):
            for b in (wb[1:68, 1:66], wb[1:68, 1:66].t().contiguous().t()):
                c = ops.gemm(a, b, out_dtype=F32).cpu().numpy()
                ref = orc.dot_general(np.ascontiguousarray(a.float().cpu().numpy()), [1], [],
                                      np.ascontiguousarray(b.float().cpu().numpy()), [0], [])
                assert rel_err(c, ref) <= 1e-4


@pytest.mark.parametrize("M,N,K", [(1000, 776, 1531), (65, 10, 33), (7, 129, 64), (256, 512, 256), (300, 2049, 40),
                                   (2049, 2051, 65), (16, 4097, 4096), (100, 1001, 4096)])
@pytest.mark.parametrize("act", [ActivationType.NONE, ActivationType.GELU])
def test_staged_epilogue_equals_unfused(cuda, M, N, K, act):
    x = synth.to_bf16_bits(synth.normal(7301, (M, K)))
    w = synth.to_bf16_bits(synth.normal(7302, (K, N), std=K ** -0.5))
    bias = synth.to_bf16_bits(synth.normal(7303, (N,), std=0.1))
    res = synth.to_bf16_bits(synth.normal(7304, (M, N)))
    BF = dtypes.BFloat16
    shapes = [make_shape(BF, *s) for s in ((M, K), (K, N), (N,), (M, N))]
    be = Backend("")
    outs = []
    for fuse in ("1", "0"):
        old = os.environ.get("GHIP_EPILOGUE_FUSION")
        os.environ["GHIP_EPILOGUE_FUSION"] = fuse
        try:
            b = be.Builder("staged")
            f = b.Main()
            p = [f.Parameter(f"p{i}", s) for i, s in enumerate(shapes)]
            f.Return([f.Add(p[3], f.FusedDense(p[0], p[1], p[2], act))])
            ex = b.Compile()
        finally:
            if old is None:
                del os.environ["GHIP_EPILOGUE_FUSION"]
            else:
                os.environ["GHIP_EPILOGUE_FUSION"] = old
        assert ("core=staged" in ex.Plan()) == (fuse == "1"), ex.Plan()
        bufs = [be.BufferFromFlatData(0, v, s) for v, s in zip((x, w, bias, res), shapes)]
        (y,) = ex.Execute(bufs)
        outs.append(be.BufferToFlatData(y).copy())
        ex.Finalize()
    assert np.array_equal(outs[0], outs[1])
    be.Finalize()
