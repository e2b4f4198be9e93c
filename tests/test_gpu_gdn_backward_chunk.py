"""GPU parity of the chunk-form Gated DeltaNet backward (triune_hip_gdn_bwd_chunked: 16-bit I/O, beta
none or per head) against the fp64 oracle, at the edges of its 64-token chunks and 16-token tiles,
through chunks too steep for the factored pair sums, and against the token-serial kernels.

Tolerance: one ULP of the gradient's type at the oracle's value (its own rounding, 1/2 ULP, with the
other half for values near a rounding boundary) plus 4e-5 of the largest gradient: the kernels work in
fp32, and a pair factor e^(G - m) e^(m - G') with exponents up to 64 carries up to
2 * 64 * 2^-24 * (1 + log2 e) = 2e-5 of relative error.
"""

import ctypes

import numpy as np
import pytest
import torch
import torch.nn.functional as F

import triune_amd.fast_gla as FG
from oracle import oracle as O
from triune_amd import _lib, fast_chunk_gated_deltanet

pytestmark = pytest.mark.gpu


def _ulp(r, dtype):
    bits, emin = (7, -126) if dtype == torch.bfloat16 else (10, -14)
    return torch.exp2(torch.floor(torch.log2(r.abs().clamp_min(2.0**emin))) - bits)


def _check(got, ref, dtype, names):
    for name, x, r in zip(names, got, ref):
        if r is None:
            assert x is None, name
            continue
        r = torch.as_tensor(np.asarray(r, dtype=np.float64))
        assert x.dtype == dtype and tuple(x.shape) == tuple(r.shape), name
        err = (x.detach().double().cpu() - r).abs()
        slack = 4e-5 * max(1.0, float(r.abs().max()))
        assert bool((err <= _ulp(r, dtype) + slack).all()), (name, float((err - _ulp(r, dtype)).max()), slack)


def _inputs(B, T, H, D, gate, beta, dtype, seed, steep=None, resets=False):
    gen = torch.Generator().manual_seed(seed)
    q, k = (F.normalize(torch.randn(B, T, H, D, generator=gen), dim=-1).to(dtype) for _ in range(2))
    v, do = (torch.randn(B, T, H, D, generator=gen).to(dtype) for _ in range(2))
    g = F.logsigmoid(torch.randn(*((B, T, H) if gate == "head" else (B, T, H, D)), generator=gen))
    g = g * (1.0 if gate == "key" else 0.2)
    g[:, 2::9] = 0.0  # on the clamp's edge: the gradient passes
    g[:, 1::7] = 0.05  # clamped: no gradient
    if steep is not None:
        g[:, : T // 2] = g[:, : T // 2] * steep  # some chunks steep, some not
        if resets:
            g[:, 5::31] = -float("inf")
    b = torch.sigmoid(torch.randn(B, T, H, generator=gen)).to(dtype) if beta else None
    ds = torch.randn(B, H, D, D, generator=gen)
    return q, k, v, g.to(dtype), b, do, ds


def _run(dev, q, k, v, g, b, do, ds):
    kind = _lib.BETA_NONE if b is None else _lib.BETA_HEAD
    args = [None if x is None else x.to(dev) for x in (q, k, v, g, b)]
    got = FG._gdn_bwd(*args, None, kind, None if do is None else do.to(dev), None if ds is None else ds.to(dev))
    torch.cuda.synchronize()
    gf = g.unsqueeze(-1).expand(*g.shape, q.shape[-1]) if g.dim() == 3 else g
    ref = list(O.gdn_bwd(q, k, v, gf, b, None, do, ds))
    if g.dim() == 3:
        ref[3] = ref[3].sum(-1)
    return got, ref


NAMES = ("dq", "dk", "dv", "dg", "dbeta")


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("T", [1, 15, 16, 63, 64, 65, 200])
@pytest.mark.parametrize("gate,beta", [("key", False), ("head", True)])
def test_chunk_edges(dev, D, T, gate, beta):
    x = _inputs(2, T, 3, D, gate, beta, torch.bfloat16, seed=T + D)
    got, ref = _run(dev, *x)
    _check(got, ref, torch.bfloat16, NAMES)


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("gate,beta", [("key", True), ("head", False)])
def test_many_chunks_fp16(dev, D, gate, beta):
    """Longer than the scan's prefetch, B * H past one XCD group, no final-state gradient."""
    q, k, v, g, b, do, _ = _inputs(3, 700, 3, D, gate, beta, torch.float16, seed=D)
    got, ref = _run(dev, q, k, v, g, b, do, None)
    _check(got, ref, torch.float16, NAMES)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("gate,beta", [("key", True), ("head", True), ("key", False)])
@pytest.mark.parametrize("steep,resets", [(1.0, True), (4.0, False), (12.0, True), (40.0, False)])
def test_steep_and_reset_gates(dev, D, gate, beta, steep, resets, dtype):
    """Chunks that decay by more than 128 nats beside ordinary ones: by tiles of at most 64 nats, by
    steeper tiles, and with -inf gates that reset the state."""
    x = _inputs(1, 230, 2, D, gate, beta, dtype, seed=D + 9, steep=steep * (1 if gate == "key" else 4), resets=resets)
    got, ref = _run(dev, *x)
    _check(got, ref, dtype, NAMES)


def test_only_the_final_state(dev):
    """No gradient of o: only the final state's."""
    q, k, v, g, b, _, ds = _inputs(2, 100, 2, 64, "key", True, torch.bfloat16, seed=4)
    got, ref = _run(dev, q, k, v, g, b, None, ds)
    _check(got, ref, torch.bfloat16, NAMES)


@pytest.mark.parametrize("D", [64, 128])
def test_gate_and_beta_repeated_over_tokens(dev, D):
    """One decay and one beta per head, expanded over the tokens (stride 0), with a partial last chunk
    and a gradient of the final state: the gates past the last token count as none."""
    q, k, v, _, _, do, ds = _inputs(2, 100, 3, D, "head", True, torch.bfloat16, seed=D)
    g = torch.tensor([-0.25, -0.03125, -0.5]).bfloat16().expand(2, 100, 3)
    b = torch.tensor([0.5, 0.25, 0.75]).bfloat16().expand(2, 100, 3)
    kind = _lib.BETA_HEAD
    dg, db = (x[0, 0].to(dev).expand(2, 100, 3) for x in (g, b))
    got = FG._gdn_bwd(*(x.to(dev) for x in (q, k, v)), dg, db, None, kind, do.to(dev), ds.to(dev))
    torch.cuda.synchronize()
    ref = list(O.gdn_bwd(q, k, v, g.unsqueeze(-1).expand(2, 100, 3, D).contiguous(), b.contiguous(), None, do, ds))
    ref[3] = ref[3].sum(-1)
    _check(got, ref, torch.bfloat16, NAMES)


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("shared", ["heads", "cut"])
def test_one_token_of_token_stride_zero(dev, D, shared):
    """One token whose rows have token stride 0 (k, v and dO shared by the heads, or cut from a tensor
    expanded over tokens), with a gradient of the final state: there are no tokens past it."""
    B, H = 2, 3
    q, k, v, g, _, do, ds = _inputs(B, 1, H, D, "key", False, torch.bfloat16, seed=D)

    def zero_stride(x):
        y = x.to(dev)
        if shared == "heads":
            y = y[:, :, :1].contiguous().view(B, D).as_strided((B, 1, H, D), (D, 0, 0, 1))
        else:
            y = y[:, :1].expand(B, 5, H, D)[:, :1]
        assert y.stride(1) == 0
        return y

    x = [zero_stride(t) for t in (q, k, v, g, do)]
    got = FG._gdn_bwd(x[0], x[1], x[2], x[3], None, None, _lib.BETA_NONE, x[4], ds.to(dev))
    torch.cuda.synchronize()
    c = [t.cpu().contiguous() for t in x]
    ref = O.gdn_bwd(c[0], c[1], c[2], c[3], None, None, c[4], ds)
    _check(got, ref, torch.bfloat16, NAMES)


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("gate,beta", [("key", False), ("head", True)])
def test_small_gate_gradients(dev, D, gate, beta):
    """dg is a difference of sums: fp32 products (2^-24 of each term, exponents up to 26 nats on either
    side of the midpoint: about 60 * 2^-24 = 4e-6) leave its elements below a thousandth of the rms
    (2^-12 of which, 2.4e-7, is fp16's own rounding) within 2e-6 of the rms, root mean square."""
    q, k, v, g, b, do, ds = _inputs(2, 600, 3, D, gate, beta, torch.float16, seed=D + 5)
    got, ref = _run(dev, q, k, v, g, b, do, ds)
    r = torch.as_tensor(np.asarray(ref[3], dtype=np.float64))
    rms = float(r.square().mean().sqrt())
    small = (r != 0) & (r.abs() < (1e-3 if gate == "key" else 2e-2) * rms)
    assert int(small.sum()) >= 20
    err = (got[3].double().cpu() - r)[small].square().mean().sqrt()
    assert float(err) <= (2e-6 if gate == "key" else 6e-6) * rms, float(err) / rms


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("gate", ["key", "head"])
@pytest.mark.parametrize("rate", [1.5, 3.0, 12.0])
def test_gate_gradients_of_steep_gates(dev, D, gate, rate):
    """Every gate near -rate (chunks in one piece, by tiles, token by token): each gate's gradient is
    about e^-rate of a token's products with itself and with the final state's gradient, which must
    cancel without leaving their rounding behind.  What is left is off by fp32's 2^-24 of up to 64 terms
    of its own size, with exponents up to 48 nats: 2^-24 (64 + 2 * 48 * log2 e) = 1.2e-5."""
    q, k, v, g, b, do, ds = _inputs(2, 130, 2, D, gate, gate == "head", torch.bfloat16, seed=D)
    g = (-rate * (1 + 0.1 * torch.rand(g.shape, generator=torch.Generator().manual_seed(D)))).bfloat16()
    got, ref = _run(dev, q, k, v, g, b, do, ds)
    r = torch.as_tensor(np.asarray(ref[3], dtype=np.float64))
    err = (got[3].double().cpu() - r).abs()
    assert bool((err <= _ulp(r, torch.bfloat16) + 1.2e-5 * float(r.abs().max())).all()), float(
        ((err - _ulp(r, torch.bfloat16)) / r.abs().max()).max())


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("T", [0, 1, 64, 150])
@pytest.mark.parametrize("ds", [True, False])
def test_entry_with_an_initial_state(dev, D, T, ds):
    """The entry itself with an initial state and its gradient (fp32: a chain of fp32 products over the
    chunks, 4e-5 of the largest as for the others), which the Python layer leaves to the other entry."""
    B, H = 2, 3
    q, k, v, g, b, do, dsf = _inputs(B, max(T, 1), H, D, "key", True, torch.bfloat16, seed=T + D)
    q, k, v, g, b, do = (x[:, :T].contiguous().to(dev) for x in (q, k, v, g, b, do))
    s0 = (0.3 * torch.randn(B, H, D, D, generator=torch.Generator().manual_seed(T))).to(dev)
    dsf = dsf.to(dev) if ds else None
    L = _lib.lib()
    dq, dk, dv, dg, db = (torch.empty_like(x) for x in (q, k, v, g, b))
    ds0 = torch.empty_like(s0)
    ws = torch.empty(int(L.triune_hip_gdn_bwd_chunked_workspace_size(B, T, H, D, D)), device=dev, dtype=torch.uint8)
    st = (ctypes.c_int64 * 18)(*([T * H * D, H * D, D] * 4), T * H, H, 1, T * H * D, H * D, D)
    # an empty tensor has no address: the entry wants one
    ptr = [x.data_ptr() or ws.data_ptr() for x in (q, k, v, g, b, do, dq, dk, dv, dg, db)]
    rc = L.triune_hip_gdn_bwd_chunked(*ptr[:4], 1, 1, 0, ptr[4], 1, _lib.BETA_HEAD, st, s0.data_ptr(), ptr[5],
                                      dsf.data_ptr() if ds else None, *ptr[6:], ds0.data_ptr(), B, T, H, D, D,
                                      ws.data_ptr(), ws.numel(), _lib.stream_of(q))
    _lib.check(rc, "gdn_bwd_chunked")
    torch.cuda.synchronize()
    if T == 0:
        assert torch.equal(ds0, dsf if ds else torch.zeros_like(s0))
        return
    ref = O.gdn_bwd(*(x.cpu() for x in (q, k, v, g, b, s0, do)), dsf.cpu() if ds else None)
    _check((dq, dk, dv, dg, db), ref[:5], torch.bfloat16, NAMES)
    r = torch.as_tensor(np.asarray(ref[5], dtype=np.float64))
    assert float((ds0.double().cpu() - r).abs().max()) <= 4e-5 * max(1.0, float(r.abs().max()))


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("steep", [1.0, 12.0])
def test_captured_backward_replays(dev, D, steep):
    """The backward captured in a graph gives the eager call's bits on every replay, with eager work in
    between and new inputs in the captured buffers."""
    q, k, v, g, b, do, ds = (x.to(dev) for x in _inputs(2, 200, 2, D, "key", True, torch.bfloat16, seed=D, steep=steep,
                                                        resets=steep > 1))
    kind = _lib.BETA_HEAD
    call = lambda: FG._gdn_bwd(q, k, v, g, b, None, kind, do, ds)  # noqa: E731
    call()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = call()
    for n in range(3):
        do.copy_(torch.randn(do.shape, generator=torch.Generator().manual_seed(n)))
        graph.replay()
        torch.cuda.synchronize()
        got = [x.clone() for x in out[:5]]
        for x, y in zip(got, call()[:5]):
            assert torch.equal(x, y)


@pytest.mark.parametrize("gate", ["key", "head"])
def test_operator_views_and_padding(dev, gate, monkeypatch):
    """The operator's autograd with strided q, k, v views, a non-contiguous beta and gate, and head
    dims 48 (padded to 64): the chunk form and the token-serial kernels give the same gradients to
    within a bf16 rounding of each."""
    gen = torch.Generator().manual_seed(8)
    B, T, H, D = 2, 150, 3, 48
    qkv = torch.randn(B, T, 3, H, D, generator=gen).to(dev)
    qkv[:, :, :2] = F.normalize(qkv[:, :, :2], dim=-1)
    qkv = qkv.bfloat16().requires_grad_()
    gw = (B, H, T) if gate == "head" else (B, H, T, D)
    g = (F.logsigmoid(torch.randn(*gw, generator=gen)) / 4).bfloat16().to(dev).requires_grad_()
    be = torch.sigmoid(torch.randn(B, H, T, generator=gen)).bfloat16().to(dev).requires_grad_()
    do = torch.randn(B, T, H, D, generator=gen).bfloat16().to(dev)
    res = []
    for on in (True, False):
        monkeypatch.setattr(FG, "_chunked_gdn_bwd_enabled", on)
        o, _ = fast_chunk_gated_deltanet(qkv[:, :, 0], qkv[:, :, 1], qkv[:, :, 2], g.transpose(1, 2),
                                         beta=be.transpose(1, 2))
        res.append(torch.autograd.grad(o, (qkv, g, be), do))
    torch.cuda.synchronize()
    for x, y in zip(*res):
        x, y = x.double().cpu(), y.double().cpu()
        # the token-serial path rounds each key dim's part of a head gate's gradient: D roundings
        slack = 4e-5 + (D**0.5 * 2.0**-9 if gate == "head" and x.dim() == 3 else 0.0)
        assert bool(((x - y).abs() <= 2 * _ulp(y, torch.bfloat16) + slack * max(1.0, float(y.abs().max()))).all())
