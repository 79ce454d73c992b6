"""Row kernels on rows of any width and element alignment (widths that are not whole
16-byte vectors, bases inside one, rows of one vector or less) and on wide softmax rows
(one 1024-thread workgroup a row), against the fp64 oracle: fp32 <= 1e-5 relative
(RMS-floored), 16-bit one rounding of it (2^-8 bf16, 2^-11 f16, plus the fp32 part)."""
import numpy as np
import pytest
import torch

from oracle import oracle as orc
from gomlx_hip import ops, synth
from conftest import rel_err

pytestmark = pytest.mark.gpu

TOL = {torch.float32: 1e-5, torch.bfloat16: 2.0 ** -8 + 1e-5, torch.float16: 2.0 ** -11 + 1e-5}
# One element; inside one vector; around the widths where the lanes, vectors a lane and
# waves a row change (256, 512, 1024, 2048, 4096, 8192 fp32); 16 K and more.
WIDTHS = [1, 2, 5, 9, 255, 257, 513, 1021, 1030, 2047, 4099, 8190, 8201, 16389]
WIDE = [20000, 32003, 65533, 65536]


def _rows(cuda, rows, n, dt, base, seed, std=2.0):
    """[rows, n] values starting `base` elements into a buffer of NaN (so values read
    from outside a row show), as (device view, fp32 host copy)."""
    buf = torch.full((rows * n + 64,), float("nan"), device=cuda, dtype=dt)
    v = buf[base:base + rows * n]
    v.copy_(synth.normal_device(seed, (rows * n,), std=std, device=cuda, dtype=dt))
    x = v.view(rows, n)
    return x, x.float().cpu().numpy()


def _out(cuda, rows, n, dt, base):
    """An output view and a check that nothing around it was written."""
    buf = torch.full((rows * n + 64,), 7.0, device=cuda, dtype=dt)

    def untouched():
        assert torch.all(buf[:base] == 7.0) and torch.all(buf[base + rows * n:] == 7.0)
    return buf[base:base + rows * n].view(rows, n), untouched


@pytest.mark.parametrize("n", WIDTHS + WIDE)
@pytest.mark.parametrize("dt", list(TOL))
@pytest.mark.parametrize("base", [0, 3])
def test_softmax(cuda, n, dt, base):
    rows = 5
    x, xh = _rows(cuda, rows, n, dt, base, 8100 + n)
    for log in (False, True):
        y, untouched = _out(cuda, rows, n, dt, base + (2 if log else 0))  # x and y aligned alike and not
        ops.softmax(x, log=log, out=y)
        ref = orc.softmax(xh, log=log) if log else orc.softmax(xh)
        assert rel_err(y.float().cpu().numpy(), ref) <= TOL[dt]
        untouched()


@pytest.mark.parametrize("n", [7, 1021])
def test_softmax_infinities(cuda, n):
    x, xh = _rows(cuda, 4, n, torch.float32, 3, 8200)
    x[1, 1:] = float("-inf")     # one finite value
    x[2] = float("-inf")         # none: NaN
    y = ops.softmax(x).cpu().numpy()
    assert y[1, 0] == 1.0 and np.all(y[1, 1:] == 0.0) and np.all(np.isnan(y[2]))
    assert rel_err(y[[0, 3]], orc.softmax(xh[[0, 3]])) <= 1e-5


@pytest.mark.parametrize("n", WIDTHS)
@pytest.mark.parametrize("dt", list(TOL))
@pytest.mark.parametrize("base", [0, 3])
@pytest.mark.parametrize("params", [(), ("gamma",), ("gamma", "beta")])
def test_norms(cuda, n, dt, base, params):
    rows = 5
    x, xh = _rows(cuda, rows, n, dt, base, 8300 + n)
    x += 0.5
    xh = x.float().cpu().numpy()
    pv = {k: _rows(cuda, 1, n, dt, 1, 8400 + i, std=1.0)[0].view(n) for i, k in enumerate(params)}
    ph = {k: v.float().cpu().numpy() for k, v in pv.items()}
    y, untouched = _out(cuda, rows, n, dt, base)
    ops.layernorm(x, pv.get("gamma"), pv.get("beta"), 1e-5, out=y)
    ref = orc.layernorm(xh, ph.get("gamma"), ph.get("beta"), 1e-5)
    if n > 1:  # one element: x - mean is 0 up to the rounding of the mean
        assert rel_err(y.float().cpu().numpy(), ref) <= 2 * TOL[dt]
    untouched()
    if "beta" not in params:
        y, untouched = _out(cuda, rows, n, dt, base)
        ops.rmsnorm(x, pv.get("gamma"), 1e-6, out=y)
        assert rel_err(y.float().cpu().numpy(), orc.rmsnorm(xh, ph.get("gamma"), 1e-6)) <= TOL[dt]
        untouched()
