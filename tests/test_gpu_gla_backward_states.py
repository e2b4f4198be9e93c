"""fast_chunk_gla's backward on the segment states its forward kept gives the same bits as the one
that recomputes them: one and several segments, padded head dims, a partial last chunk, the unclamped
one-token tail, an initial state, a second backward over the same graph, and calls whose forward keeps
nothing (the single launch, heads run in blocks)."""

import pytest
import torch

import triune_amd.fast_gla as FG
from triune_amd import fast_chunk_gla
from triune_amd.workloads import gla_inputs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,D", [(torch.bfloat16, 64), (torch.float16, 48), (torch.float32, 32), (torch.bfloat16, 128)])
@pytest.mark.parametrize("B,T,H,s0", [(1, 63, 2, True), (2, 1025, 3, False), (8, 1500, 8, True)])
def test_kept_states_match_recomputed(dev, monkeypatch, dtype, D, B, T, H, s0):
    q, k, v, g, st = gla_inputs(B, T, H, D, seed=T + D, dtype=dtype, init_std=0.1)
    xs = [x.to(dev).requires_grad_() for x in (q, k, v, g)] + ([st.to(dev).requires_grad_()] if s0 else [])
    do = torch.randn(B, T, H, D, generator=torch.Generator().manual_seed(1)).to(dtype).to(dev)
    o, s = fast_chunk_gla(*xs[:4], initial_state=xs[4] if s0 else None)
    ds = torch.ones_like(s)
    kept = torch.autograd.grad([o, s], xs, [do, ds], retain_graph=True)
    again = torch.autograd.grad([o, s], xs, [do, ds])
    plain = FG._prefill_bwd
    monkeypatch.setattr(FG, "_prefill_bwd", lambda *a, fwd_ws=None, **kw: plain(*a, **kw))
    o, s = fast_chunk_gla(*xs[:4], initial_state=xs[4] if s0 else None)
    fresh = torch.autograd.grad([o, s], xs, [do, ds])
    torch.cuda.synchronize()
    for a, b, c in zip(kept, again, fresh):
        assert torch.equal(a, b) and torch.equal(a, c)
