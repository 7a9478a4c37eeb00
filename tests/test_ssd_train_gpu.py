"""GPU parity: the backward of hmx.mamba_chunk_scan_combined (the training scan,
training/src/hmf/model/hybrid_zoo/layers/mamba/mamba2.py:555-580, under autograd)
against autograd through the fp64 CPU oracle (oracle/ssd.py, whose forward is pinned
by test_oracle_ssd.py).

The loss is a fixed random weighting of y (and of the final states when returned),
so every gradient path is exercised: x, dt (through softplus and the dt_limit
clamp), A, B, C (groups shared by several heads: atomics), D per head and per
(head, headdim), z, dt_bias and initial_states; seq_idx restarts, ragged last
chunks, sequences shorter than one chunk.  Tolerance: the backward's products take
bf16 operands (as mamba_ssm's do) with fp32 accumulation; each gradient must match
to 2% of its norm with cosine above 1 - 1e-4 (measured: 0.1-0.9%, cosine above
1 - 2e-5), far below what a dropped or mis-signed term gives.  dA is a per-head sum
over every token of dt'_t da_t whose terms can cancel (23x in the B-groups-wider
case), so its error is measured against the norm of the per-head sums of |dt'_t
da_t| (from the fp64 chunked backward of oracle/ssd_train.py) and must stay under
1% of it (measured up to 0.4%).
"""
import math

import pytest
import torch

import hmx
from oracle import ssd as ref
from oracle import ssd_train as oref

pytestmark = pytest.mark.gpu


def _inputs(b, l, H, G, P, N, seed, z, d_hdim):
    g0 = torch.Generator().manual_seed(seed)
    x = torch.randn(b, l, H, P, generator=g0).bfloat16()
    B = torch.randn(b, l, G, N, generator=g0).bfloat16()
    C = torch.randn(b, l, G, N, generator=g0).bfloat16()
    dt = torch.randn(b, l, H, generator=g0) * 0.5 - 2.0
    u = torch.rand(H, generator=g0)
    bias = ref.softplus_inverse(torch.exp(u * (math.log(0.1) - math.log(1e-3)) + math.log(1e-3)))
    A = -torch.exp(torch.rand(H, generator=g0) * math.log(16))
    D = (torch.randn(H, P, generator=g0) if d_hdim else torch.randn(H, generator=g0)) * 0.1 + 1.0
    zz = torch.randn(b, l, H, P, generator=g0).bfloat16() if z else None
    h0 = torch.randn(b, H, P, N, generator=g0) * 0.1
    wy = torch.randn(b, l, H, P, generator=g0)
    wf = torch.randn(b, H, P, N, generator=g0)
    return dict(x=x, dt=dt, A=A, B=B, C=C, D=D, dt_bias=bias, z=zz, initial_states=h0), wy, wf


def _grads(inp, wy, wf, kw, dev, dtype):
    """Gradients of sum(y * wy) (+ sum(final * wf)) through hmx (dev) or the oracle."""
    leaves = {k: (None if v is None else
                  v.to(dev if dev is not None else "cpu").to(dtype or v.dtype).requires_grad_(True))
              for k, v in inp.items()}
    args = dict(leaves)
    if dev is None:
        out = ref.mamba_chunk_scan_combined(args.pop("x"), args.pop("dt"), args.pop("A"),
                                            args.pop("B"), args.pop("C"), 256, **args, **kw)
    else:
        out = hmx.mamba_chunk_scan_combined(args.pop("x"), args.pop("dt"), args.pop("A"),
                                            args.pop("B"), args.pop("C"), 256, **args, **kw)
    y, fin = (out if isinstance(out, tuple) else (out, None))
    wy_ = wy.to(y.device, torch.float64 if dev is None else torch.float32)
    loss = (y.to(wy_.dtype) * wy_).sum()
    if fin is not None:
        loss = loss + (fin.to(wy_.dtype) * wf.to(fin.device, wy_.dtype)).sum()
    loss.backward()
    return {k: v.grad for k, v in leaves.items() if v is not None}


def _dA_scale(inp, wy, wf, kw):
    """Per head, sum over every chunk of every sequence of |dt'_t da_t| (the fp64
    chunked backward): dA is the sum of these terms, which can cancel (23x in one
    case here), so dA's rounding error is measured against this scale."""
    b, l, H, _ = inp["x"].shape
    total = torch.zeros(H, dtype=torch.float64)
    seq_idx = kw.get("seq_idx")
    for row in range(b):
        runs = [(0, l)] if seq_idx is None else ref._runs(seq_idx[row])
        for i, (s0, s1) in enumerate(runs):
            h0 = inp["initial_states"]
            h0 = h0[row] if (h0 is not None and i == 0 and s0 == 0) else None
            fin = wf[row] if (kw.get("return_final_states") and s1 == l) else None
            sl = slice(s0, s1)
            o = oref.chunk_grads(inp["x"][row, sl], inp["dt"][row, sl], inp["A"], inp["B"][row, sl],
                                 inp["C"][row, sl], D=inp["D"],
                                 z=None if inp["z"] is None else inp["z"][row, sl],
                                 dt_bias=inp["dt_bias"], h0=h0, dy=wy[row, sl], d_final=fin,
                                 dt_softplus=kw.get("dt_softplus", False),
                                 dt_limit=kw.get("dt_limit", (0.0, float("inf"))))
            total += o["A_abs"]
    return total


def _check(g, g_ref, name, tol=2e-2, scale=None):
    a = g.detach().double().cpu().flatten()
    b = g_ref.detach().double().cpu().flatten()
    assert torch.isfinite(a).all(), f"{name}: non-finite gradient"
    if scale is not None:   # a sum of cancelling terms: error against the terms' scale
        err = (a - b).norm().item() / scale.norm().item()
        print(f"  {name}: error / ||sum|dt' da|||  {err:.2e}")
        assert err <= tol * 0.5, f"{name}: error {err:.3e} of the terms' scale"
        return
    nb = b.norm().item()
    err = (a - b).norm().item() / max(nb, 1e-30)
    cos = (a @ b).item() / max(a.norm().item() * nb, 1e-30)
    print(f"  {name}: rel err {err:.2e}, cosine {cos:.7f}")
    assert err <= tol and cos >= 1 - 1e-4, f"{name}: rel err {err:.3e}, cosine {cos:.6f}"


CASES = {
    # b, l, H, G, N, z, D per headdim, seq_idx runs, initial + final states, dt_limit
    "z_groups": (2, 160, 4, 1, 128, True, False, None, False, (0.0, float("inf"))),
    "seq_idx_states": (1, 300, 4, 4, 64, False, True, [100, 37, 163], True, (0.0, float("inf"))),
    "clamp_ragged": (2, 93, 4, 2, 128, True, True, None, True, (0.004, 0.05)),
    "long_runs": (1, 1100, 4, 2, 128, True, False, [700, 1, 399], True, (0.0, float("inf"))),
}


@pytest.mark.parametrize("case", list(CASES))
def test_scan_backward_matches_oracle_autograd(dev, case):
    b, l, H, G, N, z, d_hdim, runs, states, lim = CASES[case]
    inp, wy, wf = _inputs(b, l, H, G, 64, N, 700 + len(case), z, d_hdim)
    kw = dict(dt_softplus=True, dt_limit=lim)
    if not states:
        inp["initial_states"] = None
    else:
        kw["return_final_states"] = True
    if runs is not None:
        kw["seq_idx"] = torch.cat([torch.full((n,), i, dtype=torch.int32)
                                   for i, n in enumerate(runs)])[None].expand(b, l)
    kw_dev = dict(kw)
    if runs is not None:
        kw_dev["seq_idx"] = kw["seq_idx"].to(dev)
    print(f"[ssd bwd] case={case}", flush=True)
    g = _grads(inp, wy, wf, kw_dev, dev, None)
    torch.cuda.synchronize()
    g_ref = _grads(inp, wy, wf, kw, None, torch.float64)
    assert set(g) == set(g_ref)
    sA = _dA_scale(inp, wy, wf, kw)
    for k in g_ref:
        _check(g[k], g_ref[k], f"{case} d{k}", scale=sA if k == "A" else None)


@pytest.mark.parametrize("N", [128, 64])
def test_backward_headdim_128(dev, N):
    """headdim 128 (the hybrid layers' headdim = d_state, mamba2.py:146): C shared by
    two heads, seq_idx restarts, initial and final states, D per head, no z."""
    inp, wy, wf = _inputs(1, 230, 4, 2, 128, N, 950 + N, False, False)
    kw = dict(dt_softplus=True, return_final_states=True,
              seq_idx=torch.cat([torch.zeros(150, dtype=torch.int32),
                                 torch.ones(80, dtype=torch.int32)])[None])
    kw_dev = dict(kw, seq_idx=kw["seq_idx"].to(dev))
    g = _grads(inp, wy, wf, kw_dev, dev, None)
    torch.cuda.synchronize()
    g_ref = _grads(inp, wy, wf, kw, None, torch.float64)
    sA = _dA_scale(inp, wy, wf, kw)
    for k in g_ref:
        _check(g[k], g_ref[k], f"hdim128 N={N} d{k}", scale=sA if k == "A" else None)


@pytest.mark.parametrize("P,N,H,G,l", [(64, 128, 5, 1, 130), (64, 64, 6, 2, 65), (64, 128, 3, 3, 64),
                                       (128, 128, 3, 1, 200), (128, 64, 4, 4, 1)])
def test_backward_groups_without_z(dev, P, N, H, G, l):
    """B and C grouped alike, no z (the kernel that shares C B^T and W's products over a
    group's heads): one, odd and even heads per group, whole, ragged and one-token
    chunks, restarts, D per (head, headdim) and initial and final states."""
    inp, wy, wf = _inputs(1, l, H, G, P, N, 970 + l, False, True)
    kw = dict(dt_softplus=True, return_final_states=True)
    kw_dev = dict(kw)
    if l > 100:
        kw["seq_idx"] = (torch.arange(l) >= 70).to(torch.int32)[None]
        kw_dev["seq_idx"] = kw["seq_idx"].to(dev)
    g = _grads(inp, wy, wf, kw_dev, dev, None)
    torch.cuda.synchronize()
    g_ref = _grads(inp, wy, wf, kw, None, torch.float64)
    sA = _dA_scale(inp, wy, wf, kw)
    for k in g_ref:
        _check(g[k], g_ref[k], f"groups P={P} N={N} d{k}", scale=sA if k == "A" else None)


@pytest.mark.parametrize("P,N,H,lens", [(64, 128, 2, (1400, 3, 64, 65, 900, 1)), (128, 64, 1, (30, 1100, 1)),
                                        (64, 64, 3, (64,) * 17)])
def test_backward_state_chains_cross_blocks(dev, P, N, H, lens):
    """Few heads, many chunks: the state chains run in blocks of chunks that sequences
    cross, end in and begin in (a sequence over more than two blocks, several within one,
    one-token and whole last chunks), with initial and final states."""
    inp, wy, wf = _inputs(1, sum(lens), H, 1, P, N, 990 + len(lens), False, False)
    idx = torch.cat([torch.full((n,), i, dtype=torch.int32) for i, n in enumerate(lens)])[None]
    kw = dict(dt_softplus=True, return_final_states=True)
    g = _grads(inp, wy, wf, dict(kw, seq_idx=idx.to(dev)), dev, None)
    torch.cuda.synchronize()
    kw["seq_idx"] = idx
    g_ref = _grads(inp, wy, wf, kw, None, torch.float64)
    sA = _dA_scale(inp, wy, wf, kw)
    for k in g_ref:
        _check(g[k], g_ref[k], f"blocks P={P} N={N} d{k}", scale=sA if k == "A" else None)


def test_backward_far_apart_gradient_rows(dev):
    """dy with token rows 2^26 elements apart, so that row 32 of a chunk is 2^32 bytes past
    its first (32-bit offsets would read row 0 there, and nothing for the rows between):
    the general kernel takes it; the same gradients as from contiguous rows, to the rounding
    of two kernels that each meet _check's bound."""
    l, H, P = 34, 2, 64
    inp, wy, _ = _inputs(1, l, H, 1, P, 128, 995, False, False)
    inp.pop("z")
    leaves = {k: v.to(dev).requires_grad_(True) for k, v in inp.items()}
    args = dict(leaves)
    y = hmx.mamba_chunk_scan_combined(args.pop("x"), args.pop("dt"), args.pop("A"), args.pop("B"),
                                      args.pop("C"), 256, dt_softplus=True, **args)
    dy = wy.to(dev, torch.bfloat16)
    step = 1 << 26
    far = torch.empty((l - 1) * step + H * P, dtype=torch.bfloat16, device=dev)
    far = far.as_strided((1, l, H, P), (l * step, step, P, 1))
    far.copy_(dy)
    g = torch.autograd.grad(y, list(leaves.values()), dy, retain_graph=True)
    g_far = torch.autograd.grad(y, list(leaves.values()), far)
    torch.cuda.synchronize()
    for k, a, b in zip(leaves, g_far, g):
        _check(a, b, f"far d{k}")


@pytest.mark.parametrize("P,H,HX,G,l", [(64, 6, 2, 3, 70), (64, 4, 1, 1, 130), (128, 4, 2, 2, 65),
                                        (128, 3, 1, 3, 64)])
def test_backward_x_shared_by_heads(dev, P, H, HX, G, l):
    """x heads shared by several heads, with B and C grouped alike and no z (the group
    kernel's fp32 stores of dB and dC, and its atomics into dx), within a group and over
    several, with whole and ragged last chunks."""
    from hmx.ops.ssd_train import ssd_chunk_scan_bwd
    inp, wy, _ = _inputs(1, l, H, G, P, 128, 1050 + l, False, False)
    inp["x"] = inp["x"][:, :, :HX].contiguous()
    t = {k: v[0].to(dev) if k in ("x", "dt", "B", "C") else v.to(dev)
         for k, v in inp.items() if v is not None}
    got = ssd_chunk_scan_bwd(t["x"], t["dt"], t["A"], t["B"], t["C"], t["D"], None, t["dt_bias"],
                             True, (0.0, float("inf")), [(0, l)], None, wy[0].to(dev))
    torch.cuda.synchronize()
    g = dict(zip(("x", "dt", "A", "B", "C", "D", "dt_bias"), got))
    assert all(g[k].dtype == torch.float32 for k in ("x", "B", "C"))
    g["D"] = g["D"].sum(-1)
    inp["initial_states"] = None
    ref_in = {k: v.double().requires_grad_(True) for k, v in inp.items() if v is not None}
    a = dict(ref_in)
    xx = a.pop("x").repeat_interleave(H // HX, dim=2)
    y = ref.mamba_chunk_scan_combined(xx, a.pop("dt"), a.pop("A"), a.pop("B"), a.pop("C"), 256,
                                      dt_softplus=True, **a)
    (y * wy.double()).sum().backward()
    sA = _dA_scale(dict(inp, x=inp["x"].repeat_interleave(H // HX, dim=2)), wy, None,
                   dict(dt_softplus=True))
    for k, v in ref_in.items():
        _check(g[k], v.grad, f"x heads {HX}/{H} P={P} d{k}", scale=sA if k == "A" else None)


@pytest.mark.parametrize("P,over,l", [(64, "C", 130), (64, "x", 65), (64, "xBC", 66), (128, "C", 65),
                                      (128, "x", 130)])
def test_backward_operands_constant_over_tokens(dev, P, over, l):
    """Operands expanded over the tokens (token stride 0) under a loss that pools the
    tokens (dy expanded too) and a ragged last chunk: the rows past its tokens overlap
    real ones, and count nothing.  Every gradient against the oracle's."""
    inp, wy, _ = _inputs(1, l, 4, 2, P, 128, 1010 + l, False, True)
    inp.update({k: inp[k][:, :1].expand(-1, l, -1, -1) for k in over})
    wy = wy[:, :1].bfloat16().expand(-1, l, -1, -1)
    kw = dict(dt_softplus=True)

    def grads(fn, conv):
        t = {k: conv(v).requires_grad_(True) for k, v in inp.items() if v is not None}
        a = dict(t)
        y = fn(a.pop("x"), a.pop("dt"), a.pop("A"), a.pop("B"), a.pop("C"), 256, **a, **kw)
        return dict(zip(t, torch.autograd.grad(y, list(t.values()), conv(wy))))

    def on_dev(v):      # .to() keeps no stride of 0: the token's row moved, then expanded
        if v.dim() == 4 and v.stride(1) == 0:
            return v[:, :1].to(dev).expand(-1, l, -1, -1)
        return v.to(dev)

    assert all(on_dev(inp[k]).stride(1) == 0 for k in over) and on_dev(wy).stride(1) == 0
    g = grads(hmx.mamba_chunk_scan_combined, on_dev)
    torch.cuda.synchronize()
    g_ref = grads(ref.mamba_chunk_scan_combined, lambda v: v.double())
    sA = _dA_scale(inp, wy, None, kw)
    for k in g_ref:
        _check(g[k], g_ref[k], f"over={over} P={P} d{k}", scale=sA if k == "A" else None)


@pytest.mark.parametrize("P", [64, 128])
def test_backward_dx_at_any_element(dev, monkeypatch, P):
    """The C entry takes dx at any element: two bytes past its buffer's start it is that of
    an aligned buffer (to the rounding of two kernels), and the elements around it stay."""
    from hmx import _lib
    from hmx.ops.ssd_train import ssd_chunk_scan_bwd
    T, H = 70, 2
    inp, wy, _ = _inputs(1, T, H, 1, P, 128, 1030, False, False)
    t = {k: v[0].to(dev) if k in ("x", "dt", "B", "C") else v.to(dev)
         for k, v in inp.items() if v is not None}
    args = (t["x"], t["dt"], t["A"], t["B"], t["C"], t["D"], None, t["dt_bias"], True,
            (0.0, float("inf")), [(0, T)], None, wy[0].to(dev))
    want = ssd_chunk_scan_bwd(*args)[0]
    n = T * H * P
    buf = torch.full((n + 2,), 7.0, dtype=torch.bfloat16, device=dev)
    call = _lib.call

    def shifted(name, *a):
        a = list(a)
        if name == "hmx_ssd_chunk_bwd":
            a[38] = buf.data_ptr() + 2
        return call(name, *a)

    monkeypatch.setattr(_lib, "call", shifted)
    ssd_chunk_scan_bwd(*args)
    torch.cuda.synchronize()
    _check(buf[1:n + 1].view_as(want), want, f"dx P={P}")
    assert buf[0] == 7.0 and buf[n + 1] == 7.0


def test_backward_headdim_128_with_z_raises(dev):
    inp, _, _ = _inputs(1, 64, 2, 1, 128, 64, 1, True, False)
    x = inp["x"].to(dev).requires_grad_(True)
    y = hmx.mamba_chunk_scan_combined(x, inp["dt"].to(dev), inp["A"].to(dev), inp["B"].to(dev),
                                      inp["C"].to(dev), 256, z=inp["z"].to(dev), dt_softplus=True)
    with pytest.raises(NotImplementedError, match="z gate needs headdim 64"):
        y.float().sum().backward()


@pytest.mark.parametrize("gb,gc,bf16_params", [(4, 2, False), (1, 2, False), (4, 2, True)])
def test_backward_training_layer_layout(dev, gb, gc, bf16_params):
    """The training layer's operands (mamba2.py:541-556): x and B repeated to the H
    heads, C with its own ngroups, D per head, no z (gb = 4); B groups wider than C's
    (gb = 1: B's gradient accumulates across workgroups); and dt, D, dt_bias in the
    model's bf16 (their gradients come back in bf16)."""
    inp, wy, wf = _inputs(1, 200, 4, gb, 64, 128, 900 + gb, False, False)
    g0 = torch.Generator().manual_seed(901)
    inp["C"] = torch.randn(1, 200, gc, 128, generator=g0).bfloat16()
    if bf16_params:
        for k in ("dt", "D", "dt_bias"):
            inp[k] = inp[k].bfloat16()
    inp["initial_states"] = None
    kw = dict(dt_softplus=True)
    g = _grads(inp, wy, wf, kw, dev, None)
    torch.cuda.synchronize()
    g_ref = _grads(inp, wy, wf, kw, None, torch.float64)
    assert g["C"].shape == inp["C"].shape
    assert all(g[k].dtype == inp[k].dtype for k in g)
    sA = _dA_scale(inp, wy, wf, kw)
    for k in g_ref:
        _check(g[k], g_ref[k], f"train_layout d{k}", scale=sA if k == "A" else None)
