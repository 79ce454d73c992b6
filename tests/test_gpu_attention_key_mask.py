"""Boolean masks over the keys alone (key padding), which the 16-bit attention kernels
hold as one bit per key: tiles without a kept key, of kept keys alone and mixed ones,
at tile edges, with the causal mask, per batch and per head, grouped-query decoding
rows and split key ranges, against the fp64 oracle (normwise 1e-2 bf16 / 2e-3 f16: P
and the output are each rounded once) and against the same mask expanded over the
queries, which takes the per-lane mask path (the same arithmetic: the same bits)."""
import numpy as np
import pytest
import torch

from oracle import oracle as orc
from gomlx_hip import ops, synth
from conftest import norm_err

pytestmark = pytest.mark.gpu

BF16, F16 = torch.bfloat16, torch.float16


def _qkv(B, H, Hkv, Sq, Sk, D, dt, cuda):
    return [synth.normal_device(s, (B, h, n, D), device=cuda, dtype=dt)
            for s, h, n in ((9301, H, Sq), (9302, Hkv, Sk), (9303, Hkv, Sk))]


def _keep(kind, B, Hm, Sk, cuda):
    """[B, Hm, 1, Sk] keep flags: lengths from one key to all, or runs and holes."""
    idx = torch.arange(Sk, device=cuda)
    rows = []
    for i in range(B * Hm):
        if kind == "padding":
            rows.append(idx < [1, Sk, (Sk + 1) // 2, min(Sk, 64), min(Sk, 65)][i % 5])
        else:  # holes: whole tiles missing at the start and inside, single keys kept
            k = (idx % 192 >= 128) | (idx == 3 + i)
            rows.append(k if i % 2 else k & (idx >= 64 * (i % 3)) | (idx == Sk - 1))
    return torch.stack(rows).view(B, Hm, 1, Sk)


CASES = [  # (B, H, Hkv, Sq, Sk)
    (5, 2, 2, 130, 200), (3, 4, 2, 257, 1000), (2, 2, 1, 64, 64), (4, 2, 2, 1, 63), (5, 8, 2, 1, 700),
    (3, 8, 2, 4, 1100), (1, 2, 2, 128, 2049),
]


@pytest.mark.parametrize("case", CASES)
@pytest.mark.parametrize("kind", ["padding", "holes"])
@pytest.mark.parametrize("D,dt", [(64, F16), (128, BF16), (96, BF16), (256, F16)])
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("per_head", [False, True])
def test_key_masks(cuda, case, kind, D, dt, causal, per_head):
    B, H, Hkv, Sq, Sk = case
    if causal and Sq > Sk:
        pytest.skip("causal prefill only")
    q, k, v = _qkv(B, H, Hkv, Sq, Sk, D, dt, cuda)
    keep = _keep(kind, B, H if per_head else 1, Sk, cuda)
    if causal:
        keep[..., 0] = True  # every query sees a key
    print(case, kind, D, dt, causal, per_head, flush=True)
    got = ops.sdpa_masked(q, k, v, keep, D ** -0.5, causal)
    full = ops.sdpa_masked(q, k, v, keep.expand(B, keep.shape[1], Sq, Sk).contiguous(), D ** -0.5, causal)
    if Sq > 1:
        assert torch.equal(got, full)
    ref = orc.sdpa(*(t.float().cpu().numpy() for t in (q, k, v)), scale=D ** -0.5, causal=causal,
                   mask=keep.expand(B, keep.shape[1], Sq, Sk).cpu().numpy())
    assert norm_err(got.float().cpu().numpy(), ref) <= (2e-3 if dt == F16 else 1e-2)


@pytest.mark.parametrize("Sq", [1, 200])
def test_no_kept_key_is_nan(cuda, Sq):
    q, k, v = _qkv(2, 4, 4, Sq, 300, 64, BF16, cuda)
    keep = torch.ones((2, 1, 1, 300), dtype=torch.bool, device=cuda)
    keep[1] = False
    got = ops.sdpa_masked(q, k, v, keep, 0.125, False)
    assert torch.isnan(got[1]).all() and not torch.isnan(got[0]).any()


@pytest.mark.parametrize("D,dt,causal", [(64, F16, False), (128, BF16, True), (256, F16, False), (64, BF16, True)])
@pytest.mark.parametrize("where", ["k", "v"])
@pytest.mark.parametrize("value", [float("nan"), float("inf"), float("-inf")])
@pytest.mark.parametrize("key", [70, 130, 199])
def test_non_finite_at_a_dropped_key(cuda, D, dt, causal, where, value, key):
    """A NaN or infinity at a dropped key has one effect, whatever else its 64-key tile
    keeps (70: a tile of kept and dropped keys, 130 and 199: tiles without a kept key):
    the per-lane mask's, which adds -inf to the key's score and multiplies its V by 0."""
    B, H, Sq, Sk = 2, 2, 200, 200
    q, k, v = _qkv(B, H, H, Sq, Sk, D, dt, cuda)
    (k if where == "k" else v)[0, 1, key, 3] = value
    keep = (torch.arange(Sk, device=cuda) < 66).view(1, 1, 1, Sk).expand(B, 1, 1, Sk).contiguous()
    print(D, dt, causal, where, value, key, flush=True)
    got = ops.sdpa_masked(q, k, v, keep, D ** -0.5, causal)
    full = ops.sdpa_masked(q, k, v, keep.expand(B, 1, Sq, Sk).contiguous(), D ** -0.5, causal)
    assert torch.equal(torch.isnan(got), torch.isnan(full)) and torch.equal(got.nan_to_num(), full.nan_to_num())
    assert not torch.isnan(got[1]).any() and not torch.isnan(got[0, 0]).any()
    if where == "v" and not causal:
        assert torch.isnan(got[0, 1, :, 3]).all()
