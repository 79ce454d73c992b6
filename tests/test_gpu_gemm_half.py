"""The 256 x 128 GEMM core (grids that 256 x 256 tiles leave half empty): whole tiles in
each operand layout and, with a K-contiguous A (others run the 128 x 128 core there),
edge tiles of rows and columns and contractions of partial k-tiles, against the fp64 oracle on rows and columns at tile edges, and a fused epilogue against the
unfused plan, bit for bit.  Tolerances: one rounding of a 16-bit output (half a unit in
the last place, 2^-9 of a value in bf16 and 2^-12 in f16, values up to ~5 times the
result's RMS), and for fp32 results the sum of K products of 16-bit operands, exact in
fp32, whose K roundings of 2^-24 add up to at most K^0.5 2^-24 times a few of the RMS:
2e-5 at K = 8192."""
import os

import numpy as np
import pytest
import torch

from oracle import oracle as orc
from gomlx_hip import ops, synth
from gomlx_hip.backend import Backend, dtypes, make_shape
from conftest import rel_err

pytestmark = pytest.mark.gpu

BF16, F16, F32 = torch.bfloat16, torch.float16, torch.float32


# (batch, M, N, K): whole tiles; one row / one chunk of columns past a tile; K one chunk
# past a k-tile and past three stages; batches.
@pytest.mark.parametrize("shape", [(1, 2048, 4096, 2048), (1, 2056, 2184, 4104), (1, 4096, 1288, 4160),
                                   (2, 2048, 1152, 4232), (1, 256, 32768, 2048)])
@pytest.mark.parametrize("a_t,b_t", [(False, False), (False, True), (True, False), (True, True)])
@pytest.mark.parametrize("dt,odt", [(BF16, BF16), (F16, F32)])
def test_half_tiles(cuda, shape, a_t, b_t, dt, odt):
    B, M, N, K = shape
    print(f"256 x 128 gemm {shape} a_t={a_t} b_t={b_t} {dt}->{odt}", flush=True)
    a = synth.normal_device(7501, (B, K, M) if a_t else (B, M, K), std=0.125, device=cuda, dtype=dt)
    b = synth.normal_device(7502, (B, N, K) if b_t else (B, K, N), std=0.125, device=cuda, dtype=dt)
    a, b = (a.transpose(1, 2) if a_t else a), (b.transpose(1, 2) if b_t else b)
    rows = np.unique(np.clip(np.array([0, 1, 15, 16, 127, 128, 255, 256, 1000, M - 9, M - 1]), 0, M - 1))
    cols = np.unique(np.clip(np.array([0, 7, 8, 63, 64, 127, 128, 129, 1000, N - 8, N - 1]), 0, N - 1))
    c = ops.gemm(a, b, out_dtype=odt).float().cpu().numpy()[:, rows][:, :, cols]
    an, bn = a.float()[:, rows].cpu().numpy(), b.float()[:, :, cols].cpu().numpy()
    ref = orc.dot_general(np.ascontiguousarray(an), [2], [0], np.ascontiguousarray(bn), [1], [0])
    assert rel_err(c, ref) <= {BF16: 1e-2, F32: 2e-5}[odt]


@pytest.mark.parametrize("M,N,K,b_t", [(2048, 2304, 2048, False), (2304, 2176, 2112, True)])
def test_epilogue_bitwise(cuda, M, N, K, b_t):
    """A residual added in the 256 x 128 core's epilogue equals the unfused plan."""
    x = synth.to_bf16_bits(synth.normal(7511, (M, K), std=0.125))
    w = synth.to_bf16_bits(synth.normal(7512, (N, K) if b_t else (K, N), std=0.125))
    r = synth.to_bf16_bits(synth.normal(7513, (M, N)))
    shapes = [make_shape(dtypes.BFloat16, *v.shape) for v in (x, w, r)]
    be = Backend("")
    outs = []
    for fuse in ("1", "0"):
        old = os.environ.get("GHIP_EPILOGUE_FUSION")
        os.environ["GHIP_EPILOGUE_FUSION"] = fuse
        try:
            b = be.Builder("half")
            f = b.Main()
            p = [f.Parameter(f"p{i}", s) for i, s in enumerate(shapes)]
            f.Return([f.Add(f.DotGeneral(p[0], [1], [], p[1], [1 if b_t else 0], []), p[2])])
            ex = b.Compile()
        finally:
            if old is None:
                del os.environ["GHIP_EPILOGUE_FUSION"]
            else:
                os.environ["GHIP_EPILOGUE_FUSION"] = old
        assert ("core=4w-k64" in ex.Plan()) == (fuse == "1"), ex.Plan()
        bufs = [be.BufferFromFlatData(0, v, s) for v, s in zip((x, w, r), shapes)]
        (y,) = ex.Execute(bufs)
        outs.append(be.BufferToFlatData(y).copy())
        ex.Finalize()
    assert np.array_equal(outs[0], outs[1])
    be.Finalize()
