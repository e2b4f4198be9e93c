"""The prefill's segment plans (rounds of segments, dropped segments, packed segment lengths) against the
fp64 oracle and the forced plans, at shapes on both sides of each rule: fewer (sequence, head) pairs than
slots, so many that two rounds of segments pay, more than all of them, one chunk, and packed batches whose
estimate leaves the eight-round length."""

import numpy as np
import pytest
import torch

from oracle import oracle as O
from triune_amd import _lib, fast_chunk_gla_varlen
from triune_amd.fast_gla import _prefill
from triune_amd.workloads import gla_inputs

pytestmark = pytest.mark.gpu


def _err(a, b):
    return float((torch.as_tensor(a).double().cpu() - torch.as_tensor(np.asarray(b))).abs().max())


# The last figure: rounds of resident workgroups (two per CU at D = 64, one at D = 128) the plan takes.
@pytest.mark.parametrize("B,T,H,D,rounds", [(1, 64, 1, 64, 1), (3, 3001, 8, 64, 1), (8, 520, 12, 128, 1),
                                            (6, 300, 100, 64, 2), (17, 960, 10, 128, 2), (17, 1984, 20, 64, 2)])
def test_dense_plans(dev, B, T, H, D, rounds):
    segments = int(_lib.lib().triune_hip_gla_prefill_workspace_size(B, T, H, D, D, 0)) // (B * H * (D * D + D) * 4)
    slots = torch.cuda.get_device_properties(dev).multi_processor_count * (2 if D == 64 else 1)
    assert -(-B * H * segments // slots) == rounds and (segments > 1) == (T > 64 and B * H < slots)
    q, k, v, g, s0 = gla_inputs(B, T, H, D, seed=T, dtype=torch.bfloat16, init_std=0.1)
    g = g.float()  # the three-launch form whatever the size
    x = [t.to(dev) for t in (q, k, v, g, s0)]
    out = torch.empty(B, T, H, D, device=dev, dtype=torch.float32)
    o, s = _prefill(*x, out, 0)
    o = o.clone()
    o1, s1 = _prefill(*x, out, 3 << _lib.FLAG_SEG_SHIFT)
    torch.cuda.synchronize()
    assert float((o - o1).abs().max()) <= 2e-3 and float((s - s1).abs().max()) <= 2e-3
    # the oracle on one sequence's first and last head
    for h in (0, H - 1):
        ro, rs = O.gla_fwd(*(t[-1:, :, h:h + 1] for t in (q, k, v, g)), s0[-1:, h:h + 1])
        assert _err(o[-1:, :, h:h + 1], ro) <= 2e-3 and _err(s[-1:, h:h + 1], rs) <= 2e-3


@pytest.mark.parametrize("lens,H", [([2000, 40, 900], 12), ([5000, 7000, 3333, 64, 1], 12)])
def test_packed_plans(dev, lens, H):
    D, N = 128, sum(lens)
    cu = torch.tensor([0] + list(np.cumsum(lens)), dtype=torch.int32)
    q, k, v, g, _ = gla_inputs(1, N, H, D, seed=len(lens), dtype=torch.bfloat16)
    out = torch.empty(1, N, H, D, device=dev, dtype=torch.float32)
    o, s = fast_chunk_gla_varlen(*(t.to(dev) for t in (q, k, v, g, cu)), out=out)
    torch.cuda.synchronize()
    for h in (0, H - 1):
        ro, rs = O.gla_varlen_fwd(*(t[:, :, h:h + 1] for t in (q, k, v, g)), cu)
        assert _err(o[:, :, h:h + 1].reshape(ro.shape), ro) <= 2e-3 and _err(s[:, h:h + 1], rs) <= 2e-3
