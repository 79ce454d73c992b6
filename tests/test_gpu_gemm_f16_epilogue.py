"""Generated epilogues of fp16 products: on every GEMM core, with whole and edge tiles,
the fused step gives the bits of the unfused plan (the product rounded to fp16, then the
elementwise kernel)."""
import os

import numpy as np
import pytest

from gomlx_hip import synth
from gomlx_hip.backend import ActivationType, Backend, dtypes, make_shape

pytestmark = pytest.mark.gpu


def _dense(act):
    def build(f, p, at, bt):
        return f.FusedDense(p[0], p[1], p[2], act)
    return build


def _residual(f, p, at, bt):
    return f.Add(f.DotGeneral(p[0], [0 if at else 1], [], p[1], [1 if bt else 0], []), p[2])


def _gated(f, p, at, bt):
    g, u = (f.DotGeneral(p[0], [1], [], w, [0], []) for w in p[1:3])
    return f.Mul(f.Mul(g, f.Logistic(g)), u)


# core in the plan, (M, N, K), operands transposed, graph
CASES = [("staged", (300, 2049, 40), 0, 0, _dense(ActivationType.GELU)),
         ("staged", (65, 10, 33), 0, 0, _dense(ActivationType.RELU)),
         ("small", (1544, 1672, 136), 0, 0, _dense(ActivationType.SILU)),
         ("4w-k64", (2048, 2304, 2048), 0, 1, _residual),
         ("4w-km32", (2304, 4104, 72), 0, 0, _residual),
         ("4w-km32", (2048, 2048, 128), 0, 0, _gated),
         ("4w-km32", (3080, 4096, 136), 0, 0, _dense(ActivationType.GELU)),
         ("8w-k64", (2304, 4104, 128), 0, 1, _residual),
         ("4w-mn32", (2304, 4096, 200), 1, 0, _residual)]


@pytest.mark.parametrize("core,mnk,at,bt,build", CASES)
def test_f16_epilogue_equals_unfused(cuda, core, mnk, at, bt, build):
    M, N, K = mnk
    print(f"f16 epilogue {core} {mnk} at={at} bt={bt}", flush=True)
    third = (N,) if build not in (_residual, _gated) else (K, N) if build is _gated else (M, N)
    arrays = [synth.normal(7601, (K, M) if at else (M, K)).astype(np.float16),
              synth.normal(7602, (N, K) if bt else (K, N), std=K ** -0.5).astype(np.float16),
              synth.normal(7603, third, std=K ** -0.5).astype(np.float16)]
    shapes = [make_shape(dtypes.Float16, *a.shape) for a in arrays]
    be = Backend("")
    outs = []
    for fuse in ("1", "0"):
        old = os.environ.get("GHIP_EPILOGUE_FUSION")
        os.environ["GHIP_EPILOGUE_FUSION"] = fuse
        try:
            b = be.Builder("f16")
            f = b.Main()
            f.Return([build(f, [f.Parameter(f"p{i}", s) for i, s in enumerate(shapes)], at, bt)])
            ex = b.Compile()
        finally:
            if old is None:
                del os.environ["GHIP_EPILOGUE_FUSION"]
            else:
                os.environ["GHIP_EPILOGUE_FUSION"] = old
        assert (f"core={core} " in ex.Plan()) == (fuse == "1"), ex.Plan()
        (y,) = ex.Execute([be.BufferFromFlatData(0, a, s) for a, s in zip(arrays, shapes)])
        outs.append(be.BufferToFlatData(y).view(np.uint16).copy())
        ex.Finalize()
    assert np.array_equal(outs[0], outs[1])
    be.Finalize()
