"""The token count of pool decode steps (StateSlotPool.offsets), kept by the decode kernels: every slot
of the pool counted once per step and padded rows (slots outside the pool) not at all, for the smallest
batches and for more rows than the persistent grid holds, eagerly and under graph replay."""

import pytest
import torch

from triune_amd.serving import StateSlotPool

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fused", [True, False])
@pytest.mark.parametrize("B,H,D", [(1, 1, 64), (3, 5, 32), (7, 2, 128), (500, 4, 64)])
def test_offsets_counted_once_per_step(dev, fused, B, H, D):
    gen = torch.Generator().manual_seed(B)
    pool = StateSlotPool(2, B + 2, H, D, D, device=dev)
    slots = torch.randperm(B + 2, generator=gen)[:B].int()
    if B > 2:
        slots[1], slots[2] = -1, B + 2  # padded rows
    sl = slots.to(dev)
    x = torch.randn(B, 4, H, D, generator=gen).bfloat16().to(dev)
    q, k, v, g = (t.contiguous() for t in x.unbind(1))
    g = -g.abs()

    def step(layer, **kw):
        if fused:
            return pool.fused_decode_step(layer, x, sl, use_rope=False, **kw)
        return pool.decode_step(layer, q, k, v, g, sl, **kw)

    step(1)
    step(1)
    step(0, count_tokens=False)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        step(0)
    for n in range(1, 4):
        graph.replay()
        torch.cuda.synchronize()
        want = torch.zeros(2, B + 2, dtype=torch.int64)
        ok = (slots >= 0) & (slots < B + 2)
        want[1, slots[ok].long()] = 2
        want[0, slots[ok].long()] = n
        assert torch.equal(pool.offsets.cpu(), want)
