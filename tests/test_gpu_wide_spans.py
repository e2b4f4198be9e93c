"""GLA chunks whose key dims decay by more than 64 nats: in factored form for 16-bit inputs (up to 104 nats
in the forward, 80 in the backward) and token by token past that and for fp32 outputs, side by side, in
every chunk path, against the fp64 oracle.

Tolerances.  A product of two operands in two bf16 parts is off by at most 3 * 2^-17 of its terms' sizes;
outputs, states and gradients are sums of up to 64 * 64 terms of mixed signs, and 2e-4 of the largest value
covers them.  16-bit outputs add their own rounding, one ULP.
"""

import numpy as np
import pytest
import torch
import torch.nn.functional as F

import triune_amd.fast_gla as FG
from oracle import oracle as O
from triune_amd import fast_chunk_gla, fast_chunk_gla_varlen, fused_qkv_g_prep_chunk_gla
from triune_amd.workloads import gla_inputs, ulp_bf16

pytestmark = pytest.mark.gpu


TOL = 2e-4


def _gates(B, T, H, D, dtype, seed, top, limit=104.0):
    """Per-dim rates: chunk spans from mild up to `top` nats, one dim of the last head past 128, jittered
    by token."""
    gen = torch.Generator().manual_seed(seed)
    rate = torch.rand(B, 1, H, D, generator=gen) * top / 64
    rate[:, :, 0, 0] = top / 64
    rate[:, :, -1, 1] = 150.0 / 64
    rate[:, :, 0, 2] = 0.05
    g = -rate * (0.9 + 0.2 * torch.rand(B, T, H, D, generator=gen))
    g[:, 16:32, 0, 2] = -4.4  # most of a chunk's decay (73 of 70 + 3 nats) inside 16 tokens
    g = g.to(dtype)
    spans = -F.pad(g.float(), (0, 0, 0, 0, 0, -T % 64)).reshape(B, -1, 64, H, D).sum(2)
    heads = spans.amax(-1)  # per (b, chunk, head)
    if top < limit:
        assert int(((heads > 64) & (heads < limit)).sum()) >= B  # factored past 64
    assert int((heads > limit).sum()) >= B
    return g


def _err(a, b):
    """Largest difference over the largest value."""
    b = torch.as_tensor(np.asarray(b))
    return float((torch.as_tensor(a).double().cpu() - b).abs().max() / b.abs().max().clamp_min(1e-30))


def _check_out(o, ref):
    r = torch.from_numpy(np.asarray(ref)).reshape(o.shape)
    bits = {torch.float32: 23, torch.bfloat16: 7, torch.float16: 10}[o.dtype]
    floor = 2.0**-14 if o.dtype == torch.float16 else 2.0**-126
    ulp = torch.exp2(torch.floor(torch.log2(r.abs().clamp_min(floor))) - bits)
    assert bool(((o.double().cpu() - r).abs() <= ulp + TOL * r.abs().max()).all())


@pytest.mark.parametrize("dtype,out_dtype", [(torch.bfloat16, torch.bfloat16), (torch.float16, torch.float16),
                                             (torch.bfloat16, torch.float32)])
@pytest.mark.parametrize("D", [32, 64, 128])
@pytest.mark.parametrize("onepass", [True, False])
@pytest.mark.parametrize("top", [78.0, 102.0, 120.0])
def test_prefill(dev, monkeypatch, dtype, out_dtype, D, onepass, top):
    monkeypatch.setattr(FG, "ONEPASS", onepass)
    B, T, H = 2, 330, 3
    q, k, v, _, s0 = gla_inputs(B, T, H, D, seed=D, dtype=dtype, init_std=0.1)
    g = _gates(B, T, H, D, dtype, seed=1, top=top)
    out = torch.empty(B, T, H, D, device=dev, dtype=out_dtype)
    o, s = fast_chunk_gla(*(x.to(dev) for x in (q, k, v, g, s0)), out=out)
    torch.cuda.synchronize()
    ro, rs = O.gla_fwd(q, k, v, g, s0)
    _check_out(o, ro)
    assert _err(s, rs) <= TOL


@pytest.mark.parametrize("onepass", [True, False])
@pytest.mark.parametrize("top", [78.0, 102.0, 120.0])
@pytest.mark.parametrize("scale", [1e-4, 1e-8, 1e-11])
def test_small_values(dev, monkeypatch, onepass, top, scale):
    """Values and a carried state far below 1 keep their relative accuracy through steep chunks."""
    monkeypatch.setattr(FG, "ONEPASS", onepass)
    B, T, H, D = 2, 330, 3, 64
    q, k, v, _, s0 = gla_inputs(B, T, H, D, seed=D, dtype=torch.bfloat16, init_std=1.0)
    v, s0 = (v.float() * scale).bfloat16(), s0 * scale
    g = _gates(B, T, H, D, torch.bfloat16, seed=1, top=top)
    o, s = fast_chunk_gla(*(x.to(dev) for x in (q, k, v, g, s0)))
    torch.cuda.synchronize()
    ro, rs = O.gla_fwd(q, k, v, g, s0)
    _check_out(o, ro)
    assert _err(s, rs) <= TOL


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("out_dtype", [torch.bfloat16, torch.float32])
def test_packed(dev, D, out_dtype):
    lens, H = [1, 63, 200, 130], 2
    N = sum(lens)
    cu = torch.tensor([0] + list(np.cumsum(lens)), dtype=torch.int32)
    q, k, v, _, _ = gla_inputs(1, N, H, D, seed=3, dtype=torch.bfloat16)
    g = _gates(1, N, H, D, torch.bfloat16, seed=2, top=102.0)
    out = torch.empty(1, N, H, D, device=dev, dtype=out_dtype)
    o, s = fast_chunk_gla_varlen(*(x.to(dev) for x in (q, k, v, g, cu)), out=out)
    torch.cuda.synchronize()
    ro, rs = O.gla_varlen_fwd(q, k, v, g, cu)
    _check_out(o, ro)
    assert _err(s, rs) <= TOL


@pytest.mark.parametrize("T", [256, 2100])
def test_raw_projections(dev, T):
    """Raw gates N(-0.3, 1): logsigmoid spans of about 62 nats per chunk and dim, on both sides of 64 in
    every head; 2100 tokens run the pre-processing pass and the three-launch prefill."""
    gen = torch.Generator().manual_seed(T)
    B, H, D = 2, 2, 64
    qkv = torch.randn(B, T, 3, H, D, generator=gen).bfloat16()
    g = (torch.randn(B, T, H, D, generator=gen) - 0.3).bfloat16()
    qd, gd = qkv.to(dev), g.to(dev)
    whole = T // 64 * 64
    spans = -F.logsigmoid(g[:, :whole].float()).reshape(B, -1, 64, H, D).sum(2)
    assert 0.2 < float((spans > 64).float().mean()) < 0.8  # of (chunk, head, dim)
    heads = spans.amax(-1)
    assert float(((heads > 64) & (heads < 104)).float().mean()) > 0.8  # of the chunks of a head
    o, s = fused_qkv_g_prep_chunk_gla(qd, gd, use_rope=False)
    torch.cuda.synchronize()
    pq, pk, pv = (qd[:, :, i].cpu() for i in range(3))
    pg = torch.from_numpy(O.qkv_g_prep(qkv, g, None, None)[1]).to(torch.bfloat16)  # as the scan sees it
    ro, rs = O.gla_fwd(pq, pk, pv, pg)
    ro = torch.from_numpy(ro)
    # a gate may round to either neighbour: 2^-9 of its size per token over a few tokens' memory
    assert bool(((o.double().cpu() - ro).abs() <= 2 * ulp_bf16(ro).double() + 1e-2).all())
    assert _err(s, rs) <= 1e-2


@pytest.mark.parametrize("dtype,scale", [(torch.bfloat16, 1.0), (torch.float16, 1.0), (torch.bfloat16, 1e-8),
                                         (torch.bfloat16, 1e-11), (torch.bfloat16, 1e-14)])
@pytest.mark.parametrize("D", [32, 64])
@pytest.mark.parametrize("top", [78.0, 120.0])
def test_backward(dev, dtype, scale, D, top):
    """Upstream gradients of order 1 and, as a mean-reduced loss gives, far below."""
    B, T, H = 1, 200, 3
    q, k, v, _, s0 = gla_inputs(B, T, H, D, seed=D + 1, dtype=dtype, init_std=0.1)
    g = _gates(B, T, H, D, dtype, seed=5, top=top, limit=80.0)
    gen = torch.Generator().manual_seed(6)
    do = (torch.randn(B, T, H, D, generator=gen) * scale).to(dtype)
    ds = torch.randn(B, H, D, D, generator=gen) * scale
    got = FG._prefill_bwd(*(x.to(dev) for x in (q, k, v, g, s0, do, ds)), 0, grad_dtype=torch.float32)
    torch.cuda.synchronize()
    for name, x, r in zip(("dq", "dk", "dv", "dg", "ds0"), got, O.gla_bwd(q, k, v, g, s0, do, ds)):
        assert _err(x, r) <= TOL, (name, _err(x, r))
