"""The language model (ethos_amd.model.CompressedMoEModel) on the GPU:

  - the small model (one dense block, two expert blocks) against the reference's own
    logits (tests/golden/lm_tiny.npz, CompressedMoEModel in eval mode, model.py:367-396)
    in float32 and bfloat16, and against the float32 restatement of the reference model
    (tests/torch_reference.lm_forward, pinned to those logits) with the GPU run's routing
    imposed;
  - the whole-model workload at its own size (12 expert blocks, d_model 1024, MLA 16 heads,
    vocab 100,277, 4 x 2048 tokens, bf16): finite, run-to-run identical logits, and in
    every block the expert layer's queries, routing (every row: ids and gates) and output
    (a token subset) against the oracle, on the inputs that block received."""
import json
import os

import numpy as np
import pytest
import torch

from ethos_amd.layer import EthosExpertLayer
from ethos_amd.model import CompressedMoEModel, init_random_, lm_config
from ethos_amd.workloads import make_lm_inputs
from golden_util import GOLDEN
from gpu_util import check_all_tokens, check_out, to_host
from oracle import oracle as O
from torch_reference import lm_forward

pytestmark = pytest.mark.gpu


def _nerr(a, b):
    a = torch.as_tensor(np.asarray(a.detach().float().cpu() if torch.is_tensor(a) else a), dtype=torch.float64)
    b = torch.as_tensor(np.asarray(b.detach().float().cpu() if torch.is_tensor(b) else b), dtype=torch.float64)
    return float((a - b).norm() / b.norm())


def _fixture():
    f = np.load(os.path.join(GOLDEN, "lm_tiny.npz"), allow_pickle=False)
    return f, json.loads(str(f["meta"]))


def _bf16(a):
    return torch.from_numpy(a.view(np.int16)).view(torch.bfloat16).float()


def _run(m, ids):
    """Logits and the input each expert block received."""
    inputs = {}
    hooks = [blk.mlp.register_forward_pre_hook(lambda mod, a, i=i: inputs.__setitem__(i, a[0].detach()))
             for i, blk in enumerate(m.layers) if isinstance(blk.mlp, EthosExpertLayer)]
    try:
        with torch.no_grad():
            logits = m(ids.cuda())
    finally:
        for h in hooks:
            h.remove()
    return logits, inputs


def _small(dtype):
    f, meta = _fixture()
    cfg, sd, ids = make_lm_inputs(seed=meta["seed"], batch=meta["batch"], seq=meta["seq"])
    m = CompressedMoEModel(cfg)
    m.load_state_dict(sd)
    return f, cfg, sd, ids, m.to(dtype).cuda().eval()


def test_lm_matches_reference_logits_fp32():
    f, cfg, sd, ids, m = _small(torch.float32)
    logits, inputs = _run(m, ids)
    assert logits.shape == (2, 24, cfg.vocab_size) and logits.dtype == torch.float32
    e = _nerr(logits, f["ref_logits_fp32"])
    # each expert block's routing of the input it received, against the reference's choice
    agree = {}
    for i, x in inputs.items():
        ids_i = m.layers[i].mlp.router(x.reshape(-1, cfg.d_model))[1].cpu().numpy()
        agree[i] = int(np.all(ids_i == f[f"ref_ids_fp32_{i}"], axis=-1).sum())
    print(f"lm fp32: logits normalised error {e:.2e} vs the reference; routing rows equal per block {agree} "
          f"of {ids.numel() * cfg.num_routing_heads}")
    assert e < 1e-4, e
    assert all(v == ids.numel() * cfg.num_routing_heads for v in agree.values())


def test_lm_bf16_close_to_reference_logits():
    f, cfg, sd, ids, m = _small(torch.bfloat16)
    logits, _ = _run(m, ids)
    assert logits.dtype == torch.bfloat16
    e16 = _nerr(logits, _bf16(f["ref_logits_bf16"]))
    e32 = _nerr(logits, f["ref_logits_fp32"])
    e_ref = _nerr(_bf16(f["ref_logits_bf16"]), f["ref_logits_fp32"])
    print(f"lm bf16: normalised error {e32:.2e} vs the reference's fp32 logits (the reference's own bf16 run: "
          f"{e_ref:.2e}), {e16:.2e} vs the reference's bf16 logits")
    # at least as close to the float32 logits as the reference's own bf16 run, and the two
    # bf16 runs (different rounding sequences of the same model) within twice that
    assert e32 < 3e-2 and e32 <= e_ref
    assert e16 <= 2 * e_ref


def test_lm_matches_restatement_with_imposed_routing_fp32():
    f, cfg, sd, ids, m = _small(torch.float32)
    logits, inputs = _run(m, ids)
    with torch.no_grad():
        routing = {i: m.layers[i].mlp.router(x.reshape(-1, cfg.d_model))[1].cpu() for i, x in inputs.items()}
        ref = lm_forward({k: v.float() for k, v in sd.items()}, ids, cfg, routing)
    assert _nerr(logits, ref) < 1e-4


def test_lm_whole_model_workload_full_size():
    """12 expert blocks, d_model 1024, 4 x 2048 tokens, bf16, random init (seed 0)."""
    cfg = lm_config()
    m = init_random_(CompressedMoEModel(cfg), seed=0).to(torch.bfloat16).cuda().eval()
    ids = torch.randint(0, cfg.vocab_size, (4, 2048), generator=torch.Generator().manual_seed(0))
    logits, inputs = _run(m, ids)
    logits2, _ = _run(m, ids)
    torch.cuda.synchronize()
    assert logits.shape == (4, 2048, cfg.vocab_size)
    assert bool(torch.isfinite(logits).all())
    assert torch.equal(logits.view(torch.int16), logits2.view(torch.int16)), "logits differ between two runs"
    del logits2
    assert len(inputs) == cfg.num_layers
    n = ids.numel()
    q_sub = np.arange(0, n, 4)     # 2,048 tokens for the query projection
    y_sub = np.arange(7, n, 64)    # 128 tokens for the layer output
    for i, x in sorted(inputs.items()):
        layer = m.layers[i].mlp
        xf = x.reshape(-1, cfg.d_model).contiguous()
        with torch.no_grad():
            q = layer.router.queries(xf)
            gates, ids_l = layer.router.route(xf)
            y = layer.forward_flat(xf)
        torch.cuda.synchronize()
        P = O.unpack_state({k: v.cpu() for k, v in layer.state_dict().items()}, cfg.num_routing_heads)
        xs, qh = to_host(xf), to_host(q)
        assert np.array_equal(qh[q_sub], O.query_proj(xs[q_sub], P["Wq"], P["bq"], P["alpha"], P["beta"], "bf16"))
        g_ref, ids_ref = O.route(qh, P["K1"], P["K2"], cfg.top_k, "bf16")
        ih, gh = to_host(ids_l), to_host(gates)
        rows = int(np.any(ih != ids_ref, -1).sum())
        print(f"block {i}: {rows} of {ih.shape[0] * ih.shape[1]} routing rows differ from the oracle, "
              f"{int(np.count_nonzero(gh != g_ref))} gates", flush=True)
        assert rows == 0 and np.array_equal(gh, g_ref)
        r = O.layer_forward(xs, P, cfg.num_routing_heads, cfg.top_k, "bf16", tokens=y_sub, q=qh,
                            routed=(g_ref, ids_ref))
        check_out(O.to_f32(to_host(y), "bf16")[y_sub], r["out"], "bf16", nerr_max=2e-3)
        check_all_tokens(layer, xf, gates, ids_l, y, f"block {i}")


def _attention_double(q, kv, k_rot, pos, rates, H, scale):
    """The attention of model.py:118-160 in float64 on the bf16 operands, with the rotation's own
    bf16 roundings (cosines, sines, products and sums)."""
    b, n, _ = q.shape
    ang = pos.float()[:, None] * rates
    c, s = ang.cos().bfloat16(), ang.sin().bfloat16()

    def rotate(r):
        x, y = r[..., :32], r[..., 32:]
        cc, ss = (t.view((1, n) + (1,) * (r.dim() - 3) + (32,)) for t in (c, s))
        return torch.cat((x * cc - y * ss, y * cc + x * ss), -1)

    Q, K = q.view(b, n, H, 128), kv.view(b, n, H, 128)
    qq = torch.cat((Q[..., :64], rotate(Q[..., 64:])), -1)
    kk = torch.cat((K[..., :64], rotate(k_rot).unsqueeze(2).expand(b, n, H, 64)), -1)
    d = lambda t: t.double().permute(0, 2, 1, 3).contiguous()  # noqa: E731
    S = (d(qq) @ d(kk).transpose(-1, -2).contiguous()) * scale
    S = S.masked_fill(torch.ones(n, n, dtype=torch.bool, device=q.device).triu(1), float("-inf"))
    return (torch.softmax(S, -1) @ d(K[..., 64:])).permute(0, 2, 1, 3).reshape(b, n, -1)


@pytest.mark.parametrize("b,n,H", [(1, 1, 1), (2, 31, 3), (1, 32, 2), (3, 33, 1), (1, 63, 4), (2, 64, 2), (1, 65, 5), (2, 127, 3),
                                   (1, 129, 2), (5, 130, 64), (1, 1371, 3)])
def test_mla_attention_against_float64(b, n, H):
    """The attention kernel at the edges of its tiles (32 and 64 queries, 64 keys) and both
    workgroup sizes: exponentials and results each rounded to bf16 once (2^-9 rms each at most),
    so 4e-3."""
    import math

    from ethos_amd import hip
    g = torch.Generator(device="cuda").manual_seed(n)
    rn = lambda *s: torch.randn(s, generator=g, device="cuda").bfloat16()  # noqa: E731
    q, kv, a = rn(b, n, H * 128), rn(b, n, H * 128), rn(b, n, 70)
    k_rot = a[..., 6:]
    pos = torch.randperm(3 * n, generator=g, device="cuda")[:n]
    rates = 1.0 / 10000.0 ** (torch.arange(0, 64, 2, device="cuda", dtype=torch.float32) / 64)
    scale = 1.0 / math.sqrt(128)
    o = hip.mla_attention(q, kv, k_rot, pos, rates, H, 64, 64, 64, scale)
    ref = _attention_double(q, kv, k_rot, pos, rates, H, scale)
    assert o.shape == (b, n, H * 64)
    err = float((o.double() - ref).norm() / ref.norm())
    assert err < 4e-3, err


def test_mla_attention_large_scores():
    """Scores near 10^8, whole multiples of 2^7 (so that float32 sums hold them exactly): the weights
    of earlier keys stay as they are while the maximum does, however large its rounding."""
    from ethos_amd import hip
    n, H = 500, 1
    g = torch.Generator(device="cuda").manual_seed(2)
    q, kv, k_rot = (torch.zeros(1, n, w, device="cuda").bfloat16() for w in (128, 128, 64))
    q[..., 0], q[..., 1] = 2.0 ** 14, 128.0
    kv[..., 0] = 8191.0 // 64 * 64
    kv[..., 1] = torch.randint(0, 2, (1, n), generator=g, device="cuda").bfloat16()
    kv[..., 64:] = torch.randn(1, n, 64, generator=g, device="cuda").bfloat16()
    rates = torch.ones(32, device="cuda")
    pos, scale = torch.arange(n, device="cuda"), 0.0313
    o = hip.mla_attention(q, kv, k_rot, pos, rates, H, 64, 64, 64, scale)
    s = (kv[0, :, 1].double() * 128 * scale).expand(n, n).masked_fill(torch.ones(n, n, dtype=torch.bool, device="cuda").triu(1), float("-inf"))
    ref = torch.softmax(s, -1) @ kv[0, :, 64:].double()
    # every exponential is relative to one rounded maximum, which cancels: the bound of the other sizes
    err = float((o[0].double() - ref).norm() / ref.norm())
    assert err < 4e-3, err


def test_mla_attention_scores_that_overflow():
    """Scores of the first 64 keys overflow to -inf (products of finite values): queries that also
    see later keys weigh those alone, as a softmax over all scores does; the others have no finite
    score and are NaN."""
    import math

    from ethos_amd import hip
    g = torch.Generator(device="cuda").manual_seed(1)
    n, H = 200, 2
    q, kv, k_rot = (torch.randn(1, n, w, generator=g, device="cuda").bfloat16() for w in (H * 128, H * 128, 64))
    q.view(1, n, H, 128)[..., 0] = 3e38
    kv.view(1, n, H, 128)[..., 0] = 0.0
    kv.view(1, n, H, 128)[:, :64, :, 0] = -3e38
    rates = 1.0 / 10000.0 ** (torch.arange(0, 64, 2, device="cuda", dtype=torch.float32) / 64)
    pos, scale = torch.arange(n, device="cuda"), 1.0 / math.sqrt(128)
    o = hip.mla_attention(q, kv, k_rot, pos, rates, H, 64, 64, 64, scale)
    ref = _attention_double(q, kv, k_rot, pos, rates, H, scale)
    assert torch.isnan(o[:, :64]).all()
    err = float((o[:, 64:].double() - ref[:, 64:]).norm() / ref[:, 64:].norm())
    assert err < 4e-3, err


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("rows,d,ld", [(1, 8, 8), (5, 72, 80), (33, 768, 1088), (4, 1000, 1000), (3, 2048, 2056)])
def test_rms_norm_against_float64(dt, rows, d, ld):
    """RMSNorm of strided rows: two roundings to the dtype (2^-8 and, float32, 1e-6)."""
    from ethos_amd import hip
    g = torch.Generator().manual_seed(d)
    x = (torch.randn(rows, ld, generator=g) * 3).to(dt).cuda()[:, :d]
    w = torch.randn(d, generator=g).to(dt).cuda()
    y = hip.rms_norm(x, w, 1e-6)
    ref = x.double() * torch.rsqrt(x.double().square().mean(-1, keepdim=True) + 1e-6) * w.double()
    assert y.shape == x.shape and y.is_contiguous()
    assert float((y.double() - ref).norm() / ref.norm()) < (2.0 ** -8 if dt == torch.bfloat16 else 1e-6)


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
def test_swiglu_against_float64(dt):
    from ethos_amd import hip
    g = torch.Generator().manual_seed(1)
    gu = (torch.randn(3, 7, 2 * 136, generator=g) * 4).to(dt).cuda()
    gu[0, 0, :4] = torch.tensor([90.0, -90.0, 0.0, float("inf")])
    gu[0, 0, 136:140] = 1.0
    y = hip.swiglu(gu)
    a, b = gu.double().chunk(2, -1)
    ref = a * torch.sigmoid(a) * b
    assert torch.isinf(y[0, 0, 3]) and y.shape == ref.shape
    y, ref = y.double().flatten(), ref.flatten()
    ok = torch.isfinite(ref)
    assert float((y[ok] - ref[ok]).norm() / ref[ok].norm()) < (2.0 ** -7 if dt == torch.bfloat16 else 1e-6)


def test_block_with_and_without_gradients_agree():
    """A dense block under autograd (torch operations) and without (the kernels): the same
    function to bf16 rounding, and only the first carries a graph."""
    from ethos_amd.model import TransformerBlock, lm_config
    torch.manual_seed(0)
    block = TransformerBlock(lm_config(), False).cuda().bfloat16()
    x = torch.randn(2, 97, 1024, device="cuda").bfloat16()
    pos = torch.arange(97, device="cuda")
    with torch.no_grad():
        y = block(x, None, pos)
    z = block(x, None, pos)
    assert z.grad_fn is not None
    z = z.detach()
    assert y.grad_fn is None
    assert float((y.float() - z.float()).norm() / z.float().norm()) < 1e-2


def test_blocks_on_another_device_stay_torch_operations(monkeypatch):
    """A library call goes to the current device's stream: norms, FFN and attention whose tensors
    are on another device than the current one (here: the current one taken for the second) are
    torch operations."""
    from ethos_amd import hip
    from ethos_amd.model import TransformerBlock, lm_config
    torch.manual_seed(0)
    block = TransformerBlock(lm_config(), False).cuda().bfloat16()
    x, pos = torch.randn(1, 33, 1024, device="cuda").bfloat16(), torch.arange(33, device="cuda")
    with torch.no_grad():
        y = block(x, None, pos)
        called = []
        for name in ("rms_norm", "swiglu", "mla_attention"):
            monkeypatch.setattr(hip, name, lambda *a, name=name: called.append(name))
        block(x, None, pos)
        assert set(called) == {"rms_norm", "swiglu", "mla_attention"}
        called.clear()
        monkeypatch.setattr(hip, "_current_device", lambda: 1)
        assert not hip.plain(x)
        z = block(x, None, pos)
        assert not called
    assert float((y.float() - z.float()).norm() / z.float().norm()) < 1e-2
