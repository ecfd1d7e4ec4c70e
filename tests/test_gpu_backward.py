"""Gradients of the drop-in layer against autograd through the reference's layer
(tests/torch_reference.py restates model.py:208-254 and 288-343 in float32 on the CPU).
The reference is differentiated at the expert ids the layer chose, so both differentiate
the same selection; float32 layers must agree to 1e-4 normalised error on x and every
parameter, bf16 layers to 3e-2 against the float32 reference at the bf16-rounded values."""
import numpy as np
import pytest
import torch

import ethos_amd
from ethos_amd.workloads import SHAPES, make_inputs
from torch_reference import layer_forward, leaves

pytestmark = pytest.mark.gpu


def _nerr(a: torch.Tensor, b: torch.Tensor) -> float:
    a, b = a.detach().double().cpu(), b.detach().double().cpu()
    return float((a - b).norm() / max(float(b.norm()), 1e-30))


def _grads(name, train, signal=True, hidden=False):
    sh = SHAPES[name]
    x, sd = make_inputs(sh, signal=signal)
    m = ethos_amd.EthosExpertLayer(sh.config(), hidden_space=hidden).to(sh.torch_dtype)
    m.load_state_dict(sd)
    m = m.cuda().train(train)
    xd = x.cuda().view(sh.batch, -1, sh.d_model).clone().requires_grad_(True)
    y = m(xd)
    w = torch.randn(y.shape, generator=torch.Generator().manual_seed(1)).to(y.dtype).cuda()
    (y.float() * w.float()).sum().backward()
    with torch.no_grad():
        _, ids = m.router(xd.detach().view(-1, sh.d_model))
    # the reference at the same (dtype-rounded) values, in float32
    P = leaves({k: v.to(sh.torch_dtype) for k, v in sd.items()})
    xr = x.to(sh.torch_dtype).float().clone().requires_grad_(True)
    yr, _ = layer_forward(P, xr, sh.num_heads, sh.top_k, bn_batch_stats=train, ids=ids.cpu())
    (yr * w.float().cpu().view(yr.shape)).sum().backward()
    ours = {"x": xd.grad.view(-1, sh.d_model)}
    ours.update({k: p.grad for k, p in m.named_parameters()})
    ref = {"x": xr.grad}
    ref.update({k: P[k].grad for k, _ in m.named_parameters()})
    return sh, m, y, yr, ours, ref


@pytest.mark.parametrize("name,train,hidden", [("tiny_fp32", False, False), ("tiny_fp32", True, False),
                                               ("cfg1", False, False), ("cfg1", True, False),
                                               ("tiny_fp32", True, True), ("cfg1", False, True)])
def test_grads_match_reference_fp32(name, train, hidden):
    sh, m, y, yr, ours, ref = _grads(name, train, hidden=hidden)
    assert _nerr(y.view(-1, sh.d_model), yr) < 1e-5
    for k in ref:
        assert ours[k] is not None, k
        if train and k.startswith("router.query_projs.") and k.endswith(".bias"):
            # batch-statistics BatchNorm subtracts the batch mean, so the projection bias
            # has zero gradient: both sides hold rounding noise only
            wk = k[: -len("bias")] + "weight"
            scale = float(ref[wk].norm())
            assert float(ours[k].norm()) < 1e-5 * scale and float(ref[k].norm()) < 1e-5 * scale, k
            continue
        assert ref[k] is not None and float(ref[k].norm()) > 0, k
        e = _nerr(ours[k], ref[k])
        assert e < 1e-4, (k, e)


@pytest.mark.parametrize("train", [False, True])
def test_grads_match_reference_bf16(train):
    sh, m, y, yr, ours, ref = _grads("tiny", train)
    for k in ref:
        if train and k.startswith("router.query_projs.") and k.endswith(".bias"):
            continue  # zero gradient under batch statistics (see the fp32 test)
        e = _nerr(ours[k].float(), ref[k])
        assert e < 3e-2, (k, e)
        assert ours[k].dtype == torch.bfloat16


@pytest.mark.parametrize("name", ["cfg3", "tiny_fp32"])
def test_backward_deterministic(name):
    """Two forward + backward passes of the layer on the same input give bit-identical
    gradients for x and every parameter (the expert sums have a fixed order)."""
    sh = SHAPES[name]
    x, sd = make_inputs(sh, signal=True)
    grads = []
    for _ in range(2):
        m = ethos_amd.EthosExpertLayer(sh.config()).to(sh.torch_dtype)
        m.load_state_dict(sd)
        m = m.cuda().train()
        xd = x.cuda().view(sh.batch, -1, sh.d_model).clone().requires_grad_(True)
        y = m(xd)
        w = torch.randn(y.shape, generator=torch.Generator().manual_seed(1)).to(y.dtype).cuda()
        (y.float() * w.float()).sum().backward()
        torch.cuda.synchronize()
        grads.append({"x": xd.grad.clone(), **{k: p.grad.clone() for k, p in m.named_parameters()}})
    assert grads[0].keys() == grads[1].keys()
    for k in grads[0]:
        assert torch.equal(grads[0][k], grads[1][k]), f"{name}: gradient of {k} differs between two runs"


def test_grad_path_forward_values_unchanged():
    """Autograd on or off, the forward output is the same HIP result bit for bit, and only
    the autograd pass carries a graph; BatchNorm running stats advance once per call."""
    sh = SHAPES["tiny"]
    x, sd = make_inputs(sh, signal=True)
    m = ethos_amd.EthosExpertLayer(sh.config()).to(sh.torch_dtype)
    m.load_state_dict(sd)
    m = m.cuda().eval()
    xd = x.cuda().view(sh.batch, -1, sh.d_model)
    with torch.no_grad():
        y0 = m(xd)
    y1 = m(xd.clone().requires_grad_(True))
    assert y0.grad_fn is None and y1.grad_fn is not None
    assert torch.equal(y0, y1.detach())
    scores, ids = m.router(xd.view(-1, sh.d_model).clone().requires_grad_(True))
    with torch.no_grad():
        s0, i0 = m.router(xd.view(-1, sh.d_model))
    assert scores.grad_fn is not None and torch.equal(scores.detach(), s0) and torch.equal(ids, i0)
    m.train()
    nbt = int(m.router.query_norms[0].num_batches_tracked)
    m(xd.clone().requires_grad_(True)).sum().backward()
    assert int(m.router.query_norms[0].num_batches_tracked) == nbt + 1


def test_cfg3_backward_runs_and_matches_reference_on_experts():
    """Config 3 (64 tokens, 262,144 experts, bf16): gradients of the generator weights and
    latents against the float32 reference at the layer's ids."""
    sh = SHAPES["cfg3"]
    x, sd = make_inputs(sh, signal=True)
    m = ethos_amd.EthosExpertLayer(sh.config()).to(sh.torch_dtype)
    m.load_state_dict(sd)
    m = m.cuda().eval()
    xd = x.cuda().view(1, -1, sh.d_model).clone().requires_grad_(True)
    y = m(xd)
    (y.float() ** 2).sum().backward()
    with torch.no_grad():
        _, ids = m.router(xd.detach().view(-1, sh.d_model))
    P = leaves({k: v.to(sh.torch_dtype) for k, v in sd.items()})
    xr = x.to(sh.torch_dtype).float().clone().requires_grad_(True)
    yr, _ = layer_forward(P, xr, sh.num_heads, sh.top_k, bn_batch_stats=False, ids=ids.cpu())
    (yr ** 2).sum().backward()
    for k in ("generation_network.net.0.weight", "generation_network.net.2.weight"):
        assert _nerr(dict(m.named_parameters())[k].grad.float(), P[k].grad) < 3e-2, k
    lat = m.expert_latents.weight.grad.float().cpu()
    used = np.unique(ids.cpu().numpy())
    assert _nerr(lat[used], P["expert_latents.weight"].grad[used]) < 3e-2
    unused = np.setdiff1d(np.arange(sh.num_experts), used)[:1000]
    assert float(lat[unused].abs().max()) == 0.0
    assert _nerr(xd.grad.view(-1, sh.d_model).float(), xr.grad) < 3e-2


@pytest.mark.parametrize("dt,n,H,k,dh,E,hot", [("bf16", 50, 2, 4, 64, 37, 0.0), ("bf16", 33, 8, 16, 512, 900, 0.0),
                                               ("fp32", 20, 4, 8, 96, 11, 0.0), ("bf16", 7, 3, 5, 40, 3, 0.0),
                                               ("bf16", 300, 8, 16, 512, 5000, 0.5), ("fp32", 64, 4, 8, 128, 1, 0.0)])
def test_expert_backward_entry_point(dt, n, H, k, dh, E, hot):
    """ethos_expert_backward through the C-ABI against a float64 torch evaluation of its four
    outputs (dscores, hacc, dxp, dh), on routing sorted by ethos_sort_segment: experts with
    repeated pairs, a hot expert holding half of 38,400 pairs (a segment across ~300 blocks of
    the expert-sum pass), and one expert holding every pair.  Two runs are bit-identical."""
    from ethos_amd import hip
    g = torch.Generator().manual_seed(n + dh)
    tdt = torch.bfloat16 if dt == "bf16" else torch.float32
    ids = torch.randint(0, E, (n * H * k,), generator=g, dtype=torch.int32)
    if hot > 0:
        ids[torch.rand(ids.numel(), generator=g) < hot] = 7
    seg = hip.sort_segment(ids.cuda(), E)
    U = int(seg["n_unique"].item())
    slot = seg["pair_slot"].cpu()
    h = (torch.randn(U, dh, generator=g) * 0.5).to(tdt)
    xp = torch.randn(n, dh, generator=g)
    dyb = torch.randn(n, dh, generator=g)
    gates = torch.rand(n, H, k, generator=g).to(tdt)
    dg, hacc, dxp, dhs = hip.expert_backward(h.cuda(), xp.cuda(), dyb.cuda(), seg, gates.cuda(), H, k, U)
    again = hip.expert_backward(h.cuda(), xp.cuda(), dyb.cuda(), seg, gates.cuda(), H, k, U)
    torch.cuda.synchronize()
    for a1, a2, name in zip((dg, hacc, dxp, dhs), again, ("dscores", "hacc", "dxp", "dh")):
        assert torch.equal(a1, a2), f"{name} differs between two runs"
    hd, x64, y64 = h.double(), xp.double(), dyb.double()
    t = torch.arange(n * H * k) // (H * k)
    hs = hd[slot.long()]
    c = (hs * x64[t]).sum(-1)
    act = torch.nn.functional.gelu(c)
    gp = gates.double().reshape(-1)
    da = (hs * y64[t]).sum(-1)
    cdf = 0.5 * torch.erfc(-c / 2 ** 0.5)
    dgelu = cdf + c * torch.exp(-0.5 * c * c) / (2 * torch.pi) ** 0.5
    dc = gp * dgelu * da
    a = act * gp
    ref_dg = (act * da).view(n, H, k)
    ref_hacc = torch.zeros(n, dh, dtype=torch.float64).index_add_(0, t, a[:, None] * hs)
    ref_dxp = torch.zeros(n, dh, dtype=torch.float64).index_add_(0, t, dc[:, None] * hs)
    ref_dh = torch.zeros(U, dh, dtype=torch.float64).index_add_(0, slot.long(), a[:, None] * y64[t] + dc[:, None] * x64[t])
    for got, ref, name in ((dg, ref_dg, "dscores"), (hacc, ref_hacc, "hacc"), (dxp, ref_dxp, "dxp"), (dhs, ref_dh, "dh")):
        assert got.shape == ref.shape, name
        assert _nerr(got, ref) < 1e-5, (name, _nerr(got, ref))


@pytest.mark.parametrize("dh,skip", [(96, 1), (512, 2), (40, 3)])
def test_expert_backward_takes_rows_at_any_float(dh, skip):
    """xp, dyb, the token sums and dh at addresses that are aligned to a float only: the bits of
    the aligned call."""
    from ethos_amd import hip
    from ethos_amd._lib import load
    g = torch.Generator().manual_seed(dh)
    n, H, k, E = 150, 2, 8, 300
    seg = hip.sort_segment(torch.randint(0, E, (n * H * k,), generator=g, dtype=torch.int32).cuda(), E)
    U, at = int(seg["n_unique"].item()), lambda rows: torch.zeros(rows * dh + 4, device="cuda")[skip:skip + rows * dh].view(rows, dh)
    h, gates = torch.randn(U, dh, generator=g).cuda(), torch.rand(n, H, k, generator=g).cuda()
    xp, dyb = (torch.randn(n, dh, generator=g).cuda() for _ in range(2))
    want = hip.expert_backward(h, xp, dyb, seg, gates, H, k, U)
    px, py = at(n).copy_(xp), at(n).copy_(dyb)
    assert px.data_ptr() % 16 and py.data_ptr() % 16
    dg, got = torch.empty_like(gates), [at(n), at(n), at(U)]
    ws, size = hip.workspace(load().ethos_expert_backward_workspace_bytes(n, H, k, dh), h.device)
    rc = load().ethos_expert_backward(h.data_ptr(), px.data_ptr(), py.data_ptr(), seg["pair_slot"].data_ptr(), seg["perm"].data_ptr(),
                                      seg["sorted_slot"].data_ptr(), seg["seg_off"].data_ptr(), gates.data_ptr(), n, H, k, dh, 0,
                                      ws.data_ptr(), size, dg.data_ptr(), *[t.data_ptr() for t in got], hip._stream())
    assert rc == 0
    for a, b in zip([dg] + got, want):
        assert torch.equal(a.view(b.shape), b)


@pytest.mark.parametrize("dt,n,H,k,dl,dh,d,E", [
    ("bf16", 1, 1, 1, 8, 8, 8, 1), ("bf16", 33, 2, 4, 16, 40, 72, 37), ("bf16", 129, 3, 4, 136, 264, 200, 700),
    ("bf16", 700, 4, 8, 128, 512, 256, 9000), ("bf16", 65, 8, 16, 128, 256, 1024, 1),
    # many pairs of few experts, as products
    ("bf16", 128, 8, 16, 128, 512, 64, 37), ("bf16", 130, 8, 16, 128, 256, 72, 65),
    # one pass over the experts (16,384 pairs and experts or more): one and several tiles a
    # workgroup, one and two passes of 256 columns
    ("bf16", 140, 8, 16, 128, 512, 64, 262144), ("bf16", 300, 8, 16, 128, 256, 64, 30011),
    ("bf16", 310, 8, 16, 128, 512, 64, 40000),
    ("fp32", 1, 1, 2, 8, 16, 8, 4), ("fp32", 50, 4, 8, 24, 72, 40, 11), ("fp32", 500, 4, 8, 128, 512, 256, 4096)])
def test_expert_grads_entry_point(dt, n, H, k, dl, dh, d, E):
    """ethos_expert_grads against a float64 evaluation of the same derivative: sizes off every
    tile (64, 128, 32 of the reduction), one pair, one expert, fewer unique experts than the
    buffers hold, split and unsplit reductions.  float32 sums of at most 9,000 terms: 1e-5;
    bf16 results are rounded once, at most 2^-8 of each value.  Two runs are bit-identical."""
    _check_expert_grads(dt, n, H, k, dl, dh, d, E)


@pytest.mark.parametrize("dh", [512, 256])
@pytest.mark.parametrize("distinct", [1, 37, 64, 65, 300])
def test_expert_grads_one_pass_few_experts_in_use(distinct, dh):
    """The one-pass gradients with a large table of which a reuse-heavy batch takes few experts:
    less than a tile of 64, a whole one, one row past it, and most workgroups without any."""
    _check_expert_grads("bf16", 128, 8, 16, 128, dh, 64, 20000, distinct)


def _check_expert_grads(dt, n, H, k, dl, dh, d, E, distinct=0):
    from ethos_amd import hip
    g = torch.Generator().manual_seed(n + dh + d)
    tdt = torch.bfloat16 if dt == "bf16" else torch.float32
    ids = torch.randint(0, E, (n * H * k,), generator=g, dtype=torch.int32)
    if distinct:
        pool = torch.randperm(E, generator=g)[:distinct].int()
        ids = pool[torch.randint(0, distinct, (n * H * k,), generator=g)]
    seg = hip.sort_segment(ids.cuda(), E)
    U, slot, uniq = int(seg["n_unique"].item()), seg["pair_slot"].cpu().long(), seg["uniq"].cpu().long()
    max_u = seg["uniq"].numel()
    assert not distinct or (U == distinct and max_u >= 16384)
    rn = lambda *s: torch.randn(s, generator=g).to(tdt)  # noqa: E731
    x, dy, lat = rn(n, d), rn(n, d), rn(E, dl)
    w1, w2 = (rn(dh, dl) / dl ** 0.5).to(tdt), (rn(2 * d, dh) / d ** 0.5).to(tdt)
    h = torch.zeros(max_u, dh, dtype=tdt)
    # c = h . xp of order one: gelu(c) = c (1 + erf) / 2 is good to |c| 2^-24 absolutely, so a c
    # of -5 alone (gelu 1e-6) would show as 0.3 relative, and one of -2.5 (0.016) as 1e-5
    h[:U] = (rn(U, dh) * (0.5 / dh ** 0.5)).to(tdt)
    gates = torch.rand(n, H, k, generator=g).to(tdt)
    args = [t.cuda() for t in (x, dy, h, lat, w1, w2)]
    assert hip.expert_grads_supported(*args)
    got = hip.expert_grads(*args, seg, gates.cuda(), H, k)
    again = hip.expert_grads(*args, seg, gates.cuda(), H, k)
    x64, dy64, h64, z, C, W2 = x.double(), dy.double(), h.double(), lat[uniq[:U]].double(), w1.double(), w2.double()
    A, B = W2[:d], W2[d:]
    t = torch.arange(n * H * k) // (H * k)
    xp, dyb, hs, gp = x64 @ A, dy64 @ B / H, h64[slot], gates.double().reshape(-1)
    grad = lambda v: 0.5 * torch.erfc(-v / 2 ** 0.5) + v * torch.exp(-0.5 * v * v) / (2 * torch.pi) ** 0.5  # noqa: E731
    c, da = (hs * xp[t]).sum(-1), (hs * dyb[t]).sum(-1)
    act, dc = torch.nn.functional.gelu(c), gp * grad(c) * da
    a = act * gp
    hacc = torch.zeros(n, dh, dtype=torch.float64).index_add_(0, t, a[:, None] * hs)
    dxp = torch.zeros(n, dh, dtype=torch.float64).index_add_(0, t, dc[:, None] * hs)
    dhs = torch.zeros(U, dh, dtype=torch.float64).index_add_(0, slot, a[:, None] * dyb[t] + dc[:, None] * xp[t])
    dpre = grad(z @ C.T) * dhs
    dlat = torch.zeros(E, dl, dtype=torch.float64)
    dlat[uniq[:U]] = dpre @ C
    ref = (dxp @ A.T, (act * da).view(n, H, k), dlat, dpre.T @ z, torch.cat([x64.T @ dxp, dy64.T @ hacc / H]))
    for i, name in enumerate(("dx", "dgates", "dlatents", "dw1", "dw2")):
        assert torch.equal(got[i], again[i]), f"{name} differs between two runs"
        assert got[i].shape == ref[i].shape, name
        tol = 1e-5 if dt == "fp32" or name == "dgates" else 2.0 ** -8
        assert _nerr(got[i], ref[i]) < tol, (name, _nerr(got[i], ref[i]))
    unused = torch.ones(E, dtype=torch.bool)
    unused[uniq[:U]] = False
    assert not got[2].cpu()[unused].any()


@pytest.mark.parametrize("dt", ["fp32", "bf16"])
def test_expert_grads_infinite_output_gradient(dt):
    """One infinite value of dy: its column of d W_v is the infinity times each sum of hidden
    rows, with that sum's sign, and the other columns are those of a finite dy."""
    from ethos_amd import hip
    g = torch.Generator().manual_seed(5)
    n, H, k, dl, dh, d, E = 70, 2, 4, 16, 72, 40, 50
    tdt = torch.bfloat16 if dt == "bf16" else torch.float32
    rn = lambda *s: torch.randn(s, generator=g).to(tdt)  # noqa: E731
    seg = hip.sort_segment(torch.randint(0, E, (n * H * k,), generator=g, dtype=torch.int32).cuda(), E)
    x, dy, lat, w1, w2 = rn(n, d), rn(n, d), rn(E, dl), rn(dh, dl), rn(2 * d, dh)
    h, gates = rn(seg["uniq"].numel(), dh), torch.rand(n, H, k, generator=g).to(tdt).cuda()
    args = [t.cuda() for t in (x, dy, h, lat, w1, w2)]
    plain = hip.expert_grads(*args, seg, gates, H, k)[4][d:]
    alone = torch.zeros(n, d, dtype=tdt, device="cuda")
    alone[31, 9] = 1.0
    sign = torch.sign(hip.expert_grads(args[0], alone, *args[2:], seg, gates, H, k)[4][d + 9].float())
    assert int((sign > 0).sum()) > 10 and int((sign < 0).sum()) > 10
    args[1][31, 9] = float("inf")
    got = hip.expert_grads(*args, seg, gates, H, k)[4][d:]
    assert torch.equal(got[9].float(), sign * float("inf"))
    rest = torch.arange(d, device="cuda") != 9
    assert torch.equal(got[rest], plain[rest])


@pytest.mark.parametrize("dt,n,d,H,dq,K,k,batch", [
    ("bf16", 2, 8, 1, 8, 3, 1, True), ("bf16", 37, 72, 3, 96, 37, 5, True), ("bf16", 300, 200, 2, 272, 64, 32, False),
    ("bf16", 1100, 256, 8, 512, 512, 16, True), ("fp32", 1, 8, 2, 16, 2, 2, False), ("fp32", 129, 40, 4, 64, 65, 9, True),
    ("fp32", 500, 256, 4, 256, 64, 8, True), ("fp32", 4200, 16, 1, 8, 5, 2, True),
    ("bf16", 2, 72, 3, 96, 37, 5, True), ("fp32", 2, 40, 4, 64, 65, 9, True), ("fp32", 3, 40, 2, 32, 16, 4, True)])
def test_gate_grads_entry_point(dt, n, d, H, dq, K, k, batch):
    """ethos_gate_grads against autograd in float64 through the same function, with batch and
    with running statistics: one token, lanes of 1 to 8 query values, sub-keys shared by a
    row's pairs, row chunks and splits off their sizes.  float32 queries of d terms, each
    gradient a sum of up to n H k float32 terms: 3e-5 (the softmax turns a query's absolute
    error into a relative one); bf16 results are rounded once, 2^-8.  With batch statistics of two or
    three tokens the gradients through the normalised queries are what is left where terms of the
    size that they have with constant statistics cancel (at two tokens nearly all: a query is +-1
    there): float32 roundings of those terms, 2^-17 of them, come on top.  Two runs are
    bit-identical."""
    from ethos_amd import hip
    g = torch.Generator().manual_seed(n + dq)
    tdt = torch.bfloat16 if dt == "bf16" else torch.float32
    rn = lambda *s: torch.randn(s, generator=g).to(tdt)  # noqa: E731
    x, wq, bq, k1, k2 = rn(n, d), (rn(H, dq, d) / d ** 0.5).to(tdt), rn(H, dq), rn(K, dq // 2), rn(K, dq // 2)
    k1, k2 = (k1 / dq ** 0.5).to(tdt), (k2 / dq ** 0.5).to(tdt)
    gamma, beta = (1 + 0.1 * rn(H, dq)).to(tdt), rn(H, dq)
    mean, var = rn(H, dq), (rn(H, dq).abs() + 0.5).to(tdt)
    ids = torch.randint(0, K * K, (n, H, k), generator=g, dtype=torch.int32)
    dg = torch.randn(n, H, k, generator=g)
    assert hip.gate_grads_supported(n, d, H, dq, K, k)
    heads = lambda t: [v.cuda() for v in t]  # noqa: E731
    args = [t.cuda() for t in (x, ids, dg, wq, bq, k1, k2)] + [heads(gamma), heads(beta)]
    args += [None, None] if batch else [heads(mean), heads(var)]
    got = hip.gate_grads(*args, 1e-5)
    again = hip.gate_grads(*args, 1e-5)
    P = [t.double().requires_grad_(True) for t in (x, wq, bq, gamma, beta, k1, k2)]
    X, W, B, G, Be, K1, K2 = P
    q = torch.einsum("nd,hqd->nhq", X, W) + B
    mu, va = (q.mean(0), q.var(0, unbiased=False)) if batch else (mean.double(), var.double())
    i = ids.long()

    def grads(m, v):
        y = (q - m) / torch.sqrt(v + 1e-5) * G + Be
        s = (y[:, :, None, :dq // 2] * K1[i // K]).sum(-1) + (y[:, :, None, dq // 2:] * K2[i % K]).sum(-1)
        return torch.autograd.grad(torch.softmax(s, -1), P, dg.double(), retain_graph=True)

    ref, terms = grads(mu, va), grads(mu.detach(), va.detach())
    for a, b, r, t, name in zip(got, again, ref, terms, ("dx", "dwq", "dbq", "dgamma", "dbeta", "dk1", "dk2")):
        assert torch.equal(a, b), f"{name} differs between two runs"
        assert a.dtype == tdt and a.shape == r.shape
        if (name == "dbq" and batch) or (k == 1):
            assert float(a.float().abs().max()) <= 1e-5 * max(1.0, float(ref[1].abs().max())), name  # exactly zero gradient
            continue
        tol = 3e-5 if dt == "fp32" else 2.0 ** -8
        if n <= 3 and batch and name in ("dx", "dwq"):
            assert float((a.double().cpu() - r).norm()) < tol * float(r.norm()) + 2.0 ** -17 * float(t.norm()), name
            continue
        assert _nerr(a, r) < tol, (name, _nerr(a, r))


@pytest.mark.parametrize("dt,n,H,dq,track", [("bf16", 2, 1, 4, True), ("fp32", 33, 3, 20, True), ("fp32", 5000, 2, 256, True),
                                             ("bf16", 4097, 8, 256, True), ("fp32", 70, 5, 64, False)])
def test_query_bn_train_entry_point(dt, n, H, dq, track):
    """ethos_query_bn_train against BatchNorm in float64: normalised queries and running
    statistics within one rounding of the layer's dtype (2^-8 and, float32, 1e-6)."""
    from ethos_amd import hip
    g = torch.Generator().manual_seed(n)
    tdt = torch.bfloat16 if dt == "bf16" else torch.float32
    v = (torch.randn(n, H, dq, generator=g) * 2 + 3).to(tdt)
    gamma, beta, mean = (torch.randn(H, dq, generator=g).to(tdt) for _ in range(3))
    var = torch.rand(H, dq, generator=g).to(tdt)
    m, s = ([t.cuda().clone() for t in u] for u in (mean, var))
    q = hip.query_bn_train(v.cuda(), [t.cuda() for t in gamma], [t.cuda() for t in beta], m if track else None,
                           s if track else None, 0.1, 1e-5)
    V = v.double()
    mu, va = V.mean(0), V.var(0, unbiased=False)
    tol = 2.0 ** -8 if dt == "bf16" else 1e-6
    assert _nerr(q, (V - mu) / torch.sqrt(va + 1e-5) * gamma.double() + beta.double()) < tol
    if track:
        assert _nerr(torch.stack(m), 0.9 * mean.double() + 0.1 * mu) < tol
        assert _nerr(torch.stack(s), 0.9 * var.double() + 0.1 * va * n / (n - 1)) < tol


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
def test_bn_coefficients_match_host(dt):
    """The device's eval-mode BatchNorm coefficients are the host's, bit for bit."""
    from ethos_amd import hip
    from ethos_amd.layer import _bn_eval_coefficients
    g = torch.Generator().manual_seed(0)
    norms = [torch.nn.BatchNorm1d(520) for _ in range(3)]
    for m in norms:
        m.weight.data.copy_(torch.randn(520, generator=g))
        m.bias.data.copy_(torch.randn(520, generator=g) * 3)
        m.running_mean.copy_(torch.randn(520, generator=g))
        m.running_var.copy_(torch.rand(520, generator=g) * 10.0 ** torch.randint(-6, 6, (520,), generator=g))
        m.to(dt)
    want = [np.stack(c) for c in zip(*[_bn_eval_coefficients(m, 520) for m in norms])]
    d = [m.cuda() for m in norms]
    got = hip.bn_coefficients([m.weight.detach() for m in d], [m.bias.detach() for m in d], [m.running_mean for m in d],
                              [m.running_var for m in d], norms[0].eps, 520, dt, torch.device("cuda", 0))
    for a, b in zip(got, want):
        assert np.array_equal(a.cpu().numpy(), b)


@pytest.mark.parametrize("name", ["tiny_fp32", "tiny"])
def test_backward_after_inference_mode(name):
    """What a call under torch.inference_mode packs serves a later call with gradients, in eval
    and in training mode, and with the model in another dtype than its input."""
    sh = SHAPES[name]
    x, sd = make_inputs(sh, signal=True)
    xd = x.cuda().view(sh.batch, -1, sh.d_model)
    other = torch.float32 if sh.torch_dtype == torch.bfloat16 else torch.bfloat16
    for train, dt in ((False, sh.torch_dtype), (True, sh.torch_dtype), (False, other)):
        grads = []
        for first in (False, True):
            m = ethos_amd.EthosExpertLayer(sh.config()).to(sh.torch_dtype)
            m.load_state_dict(sd)
            m = m.cuda().train(train)
            if first:
                with torch.inference_mode():
                    m.eval()(xd.to(dt))
                    m.train(train)
            y = m(xd.to(dt))
            y.float().square().sum().backward()
            grads.append([p.grad for p in m.parameters()])
        for a, b in zip(*grads):
            assert torch.equal(a, b)


@pytest.mark.parametrize("train", [False, True])
def test_router_second_derivative(train):
    """The scores' gradient can be differentiated again: create_graph gives the derivative of
    gate_path's torch operations, for x and the sub-keys."""
    sh = SHAPES["tiny_fp32"]
    x, sd = make_inputs(sh, signal=True)
    m = ethos_amd.EthosExpertLayer(sh.config())
    m.load_state_dict(sd)
    r = m.cuda().train(train).router
    xd = x.cuda().requires_grad_(True)
    scores, ids = r(xd)
    w = torch.randn(scores.shape, generator=torch.Generator().manual_seed(2)).cuda()
    leaves_ = [xd, r.sub_keys_1.weight]
    first = torch.autograd.grad((scores * w).sum(), leaves_, create_graph=True)
    second = torch.autograd.grad(sum((t ** 2).sum() for t in first), leaves_)
    ref1 = torch.autograd.grad((r.gate_path(xd, ids) * w).sum(), leaves_, create_graph=True)
    ref2 = torch.autograd.grad(sum((t ** 2).sum() for t in ref1), leaves_)
    for a, b in zip(first + second, ref1 + ref2):
        assert _nerr(a, b) < 1e-5


@pytest.mark.parametrize("train", [False, True])
def test_router_second_derivative_of_shared_parameters(train):
    """Two heads with one projection, one table for both sub-key halves, and rows that are
    themselves computed from a parameter of the router: create_graph counts each use once, as
    torch's own graph of gate_path does."""
    sh = SHAPES["tiny_fp32"]
    x, sd = make_inputs(sh, signal=True)
    m = ethos_amd.EthosExpertLayer(sh.config())
    m.load_state_dict(sd)
    r = m.cuda().train(train).router
    r.query_projs[1] = r.query_projs[0]
    r.sub_keys_2 = r.sub_keys_1
    leaves_ = [r.query_projs[0].weight, r.query_projs[0].bias, r.sub_keys_1.weight, r.query_norms[0].weight]
    w = torch.randn(sh.n_tok, sh.num_heads, sh.top_k, generator=torch.Generator().manual_seed(2)).cuda()
    both = []
    for own in (True, False):
        xd = x.cuda() * (1.0 + r.sub_keys_1.weight.mean())
        with torch.no_grad():
            _, ids = r(xd)
        s = r(xd)[0] if own else r.gate_path(xd, ids)
        first = torch.autograd.grad((s * w).sum(), leaves_, create_graph=True)
        both.append(first + torch.autograd.grad(sum((t ** 2).sum() for t in first), leaves_, retain_graph=True))
    # a projection's bias has no gradient under batch statistics: rounding alone on both sides
    for i, (a, b) in enumerate(zip(*both)):
        if not (train and i % 4 == 1):
            assert _nerr(a, b) < 1e-5, i


@pytest.mark.parametrize("n,H,dq", [(2, 8, 256), (500, 8, 256), (1024, 16, 256), (1025, 16, 256), (2048, 8, 256), (2049, 8, 256),
                                    (4096, 8, 256), (8192, 3, 256), (8193, 8, 256), (700, 4, 512), (3000, 5, 512),
                                    (33, 4, 128)])
def test_training_queries_are_per_head_batch_norms(n, H, dq):
    """bf16 training-mode queries and running statistics are those of statistics taken a head at
    a time, bit for bit, whatever number of heads shares a reduction."""
    import ethos_amd
    from ethos_amd import hip
    from ethos_amd.model import lm_config
    torch.manual_seed(n + H)
    r = ethos_amd.EthosExpertLayer(lm_config(d_model=64, num_experts=64, top_k=2, num_routing_heads=H, d_query=dq, d_latent=8,
                                             d_intermediate_hypernet=16)).to(torch.bfloat16).cuda().train().router
    x = torch.randn(n, 64, device="cuda").to(torch.bfloat16)
    with torch.no_grad():
        q = r.queries(x)
        v = hip.query_proj(x, *r._packed_weights(x.dtype, x.device)[:2], *r._identity, prepared=r._wq_prepared)
        pairs = [torch.var_mean(v[:, h].float(), 0, unbiased=False) for h in range(H)]
        norms = list(r.query_norms)
        mean, var = [torch.zeros_like(m.running_mean) for m in norms], [torch.ones_like(m.running_var) for m in norms]
        ref = hip.query_bn_train(v, [m.weight.detach() for m in norms], [m.bias.detach() for m in norms], mean, var, norms[0].momentum,
                                 norms[0].eps, batch=([p[1] for p in pairs], [p[0] for p in pairs]))
    assert torch.equal(q, ref)
    for m, a, b in zip(norms, mean, var):
        assert torch.equal(m.running_mean, a) and torch.equal(m.running_var, b)


@pytest.mark.parametrize("name", ["tiny_fp32", "tiny"])
def test_training_sees_weights_written_without_a_version_step(name):
    """A training pass, and the first evaluation after one, read the parameters as they are, also
    where an optimizer wrote them through `.data`: outputs and gradients are those of a new module
    with the same values."""
    sh = SHAPES[name]
    x, sd = make_inputs(sh, signal=True)
    xd = x.cuda().view(sh.batch, -1, sh.d_model)

    def new(state, train):
        m = ethos_amd.EthosExpertLayer(sh.config()).to(sh.torch_dtype)
        m.load_state_dict(state)
        return m.cuda().train(train)

    def step(m):
        m.zero_grad()
        y = m(xd)
        y.float().square().sum().backward()
        return [y.detach()] + [p.grad.clone() for p in m.parameters()]

    m = new(sd, True)
    step(m)
    for _ in range(2):
        versions = [p._version for p in m.parameters()]
        for p in m.parameters():
            p.data.mul_(1.25)
        assert versions == [p._version for p in m.parameters()]
        state = {k: v.clone() for k, v in m.state_dict().items()}
        for a, b in zip(step(m), step(new(state, True))):
            assert torch.equal(a, b)
    for p in m.parameters():
        p.data.mul_(0.75)
    with torch.no_grad():
        assert torch.equal(m.eval()(xd), new(m.state_dict(), False)(xd))


@pytest.mark.parametrize("H,dq", [(1, 256), (4, 256), (5, 256), (8, 256), (16, 256), (32, 256), (3, 512), (8, 512), (7, 512), (6, 64)])
def test_training_statistics_over_row_counts(H, dq):
    """The same over row counts on both sides of every line of the rule that lets heads share a
    reduction, and between them: the order of sums inside torch's reduction is not ours, and this
    sweep is what says that grouping leaves it as it is."""
    from ethos_amd.model import lm_config
    torch.manual_seed(H + dq)
    r = ethos_amd.EthosExpertLayer(lm_config(d_model=8, num_experts=64, top_k=2, num_routing_heads=H, d_query=dq, d_latent=8,
                                             d_intermediate_hypernet=16)).to(torch.bfloat16).cuda().train().router
    g = torch.Generator().manual_seed(dq)
    lines = [1 << e for e in range(1, 15)]
    ns = sorted({n + i for n in lines for i in (-1, 0, 1)} | {int(2 ** (1 + 13.3 * torch.rand(1, generator=g))) for _ in range(24)})
    seen = []

    def record(v, *a, batch=None, **k):
        seen.append((v, batch))
        return v

    from ethos_amd import hip
    was, hip.query_bn_train = hip.query_bn_train, record
    try:
        for n in ns:
            if n > 1:
                with torch.no_grad():
                    r.queries(torch.randn(n, 8, device="cuda").bfloat16() * 3 + 1)
                v, (mean, var) = seen.pop()
                for h in range(H):
                    s, m = torch.var_mean(v[:, h].float(), 0, unbiased=False)
                    assert torch.equal(mean[h], m) and torch.equal(var[h], s), (n, h)
    finally:
        hip.query_bn_train = was


def test_training_queries_of_heads_that_share_a_norm():
    """Two heads with one BatchNorm module: normalised by their own batches, and the running
    statistics updated twice, in the heads' order, as by batch_norm a head at a time."""
    from ethos_amd import hip
    sh = SHAPES["tiny_fp32"]
    x, sd = make_inputs(sh, signal=True)
    m = ethos_amd.EthosExpertLayer(sh.config())
    m.load_state_dict(sd)
    r, x = m.cuda().train().router, x.cuda()
    r.query_norms[1] = r.query_norms[0]
    norms = list(r.query_norms)
    mean, var = norms[0].running_mean.clone(), norms[0].running_var.clone()
    with torch.no_grad():
        q = r.queries(x)
        v = hip.query_proj(x, *r._packed_weights(x.dtype, x.device)[:2], *r._identity)
        for h in range(2):
            ref = torch.nn.functional.batch_norm(v[:, h], mean, var, norms[0].weight, norms[0].bias, True, 0.1, norms[0].eps)
            assert torch.equal(q[:, h], ref)
    assert torch.equal(norms[0].running_mean, mean) and torch.equal(norms[0].running_var, var)
    assert int(norms[0].num_batches_tracked) == int(sd["router.query_norms.0.num_batches_tracked"] if
                                                    "router.query_norms.0.num_batches_tracked" in sd else 0) + 2
