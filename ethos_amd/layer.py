"""Drop-in ETHOS expert layer for MI355X.

The module tree, constructor, state_dict keys and forward signatures are those of
the reference (wrmedford/ETHOS):

  ExpertGenerationNetwork(d_latent, d_model, d_intermediate)    model.py:168-179
  ProductKeyRouter(config).forward(x_flat) -> (scores, indices)  model.py:182-254
  SimplifiedHypernetMoE(config).forward(x) -> y                  model.py:267-343
  FusedLowRankMoE_Reordered(config).forward(x) -> y              kernels.py:123-221

so ``from ethos_amd import FusedLowRankMoE_Reordered`` replaces the reference import
at model.py:352 and a reference state_dict loads unchanged.  The constructor reads
config.d_model, num_experts (a perfect square), top_k, num_routing_heads, d_latent,
d_intermediate_hypernet and d_query.

Forward runs five HIP stages on the current stream (include/ethos_hip.h): query
projection + BatchNorm, product-key routing, reordering by expert id, expert
generation over the unique experts, and apply + scatter-back.  Inputs must be HIP
tensors; there is no CPU path.

With autograd enabled (the input or a parameter requires grad, outside torch.no_grad)
the output carries a graph whose gradients are those of the reference's pure-PyTorch
layer (model.py:288-343, differentiated by autograd there): through the routing gates
to the query projections, BatchNorm affine parameters and sub-keys (the topk values
and softmax, model.py:215-234), and through the generated experts to x, the expert
latents and both generator weights.  The forward values are the HIP kernels' in both
cases; the reference's Triton layer (kernels.py:145-221) has no backward at all.
"""
from __future__ import annotations

import contextlib
import math
from typing import NamedTuple

import numpy as np
import torch
import torch.nn as nn
import torch.nn.functional as F

from . import hip


def _bn_eval_coefficients(m: nn.BatchNorm1d, n: int):
    """fp32 coefficients of eval-mode BatchNorm, y = alpha * q + beta (model.py:200-202,216):
    alpha = fp32(w / sqrt(var + eps)), beta = fp32(b - mean * alpha), each evaluated in
    fp64 from the fp32 parameters and rounded once, so the result does not depend on
    which library performs the arithmetic."""
    f64 = lambda t: t.detach().float().cpu().numpy().astype(np.float64)  # noqa: E731
    w = f64(m.weight) if m.affine else np.ones(n)
    b = f64(m.bias) if m.affine else np.zeros(n)
    if m.track_running_stats and m.running_mean is not None:
        mu, var = f64(m.running_mean), f64(m.running_var)
    else:
        mu, var = np.zeros(n), np.ones(n)
    alpha = (w / np.sqrt(var + float(m.eps))).astype(np.float32)
    beta = (b - mu * alpha.astype(np.float64)).astype(np.float32)
    return alpha, beta


@contextlib.contextmanager
def _packing():
    """Around the making of what is kept between calls: ordinary tensors without a graph, also where
    the call that makes them runs under torch.inference_mode (a later one may save them for a
    backward)."""
    with torch.inference_mode(False), torch.no_grad():
        yield


class _Kept:
    """A value with tensors that is made once and read by later calls of any thread, on any stream:
    another stream's first call waits for the making and holds the memory from then on.  `once`: the
    key is that of a single pass, which goes on using the value on its stream.  What a graph capture
    makes exists only after a replay, so it is not kept for calls outside.  A copied or unpickled
    module makes its own."""

    def __init__(self):
        self.entry = None  # (key, value, event, the raw streams that are past it, tensors), replaced whole

    def get(self, key):
        entry = self.entry
        if entry is None or entry[0] != key:
            return None
        _, value, event, streams, tensors = entry
        if event is not None:
            s = hip._stream()
            # (a capture starts after the work before it: torch.cuda.graph waits for the device)
            if s not in streams and not torch.cuda.is_current_stream_capturing():
                stream = torch.cuda.current_stream()
                stream.wait_event(event)
                for t in tensors:
                    t.record_stream(stream)
                streams.add(s)
        return value

    def put(self, key, value, tensors, once: bool = False):
        on = [t for t in tensors if t is not None and t.is_cuda]
        event = None
        if on and not once:
            if torch.cuda.is_current_stream_capturing():
                return value
            event = torch.cuda.Event()
            event.record()
        self.entry = (key, value, event, {hip._stream()} if event is not None else None, on)
        return value

    def clear(self) -> None:
        self.entry = None

    @property
    def value(self):
        entry = self.entry
        return None if entry is None else entry[1]

    def __reduce__(self):
        return _Kept, ()


class _Weights(NamedTuple):
    """The routing's packed parameters in one dtype on one device."""

    wq: torch.Tensor
    bq: torch.Tensor
    k1: torch.Tensor
    k2: torch.Tensor
    key_norms: torch.Tensor
    keys_prepared: torch.Tensor | None  # the sub-keys in the scoring MFMAs' fragment order
    wq_prepared: torch.Tensor | None    # bf16: the projection weights' digit planes


def _gelu_grad(x: torch.Tensor) -> torch.Tensor:
    """Derivative of the erf GELU x·Φ(x): Φ(x) + x·φ(x)."""
    cdf = 0.5 * (1.0 + torch.erf(x * (1.0 / math.sqrt(2.0))))
    pdf = torch.exp(-0.5 * x * x) * (1.0 / math.sqrt(2.0 * math.pi))
    return cdf + x * pdf


def _gate_values(x_flat, ids, w_list, b_list, gammas, betas, k1, k2, stats, epss) -> torch.Tensor:
    """float32 gates [n, H, k] at the chosen expert ids by torch operations: per-head lists of the
    projection and BatchNorm parameters (gamma and beta None: not affine), `stats` per head
    None for batch statistics or (running mean, running variance)."""
    f = torch.float32
    H, dq, K = len(w_list), w_list[0].shape[0], k1.shape[0]
    n = x_flat.shape[0]
    w = torch.stack(w_list).to(f).reshape(H * dq, -1)
    b = torch.stack(b_list).to(f).reshape(-1)
    q = x_flat.to(f) @ w.T + b                                       # [n, H dq]
    # the H per-head BatchNorms as one over H dq channels (same per-channel statistics)
    batch = [s is None for s in stats]
    if (all(batch) or not any(batch)) and len(set(epss)) == 1:
        cat = lambda ts: torch.cat([t.to(f) for t in ts])  # noqa: E731
        affine = all(t is not None for t in gammas)
        q = F.batch_norm(q, None if batch[0] else cat(s[0] for s in stats), None if batch[0] else cat(s[1] for s in stats),
                         cat(gammas) if affine else None, cat(betas) if affine else None, batch[0], 0.0, epss[0])
    else:  # heads in different modes or with different eps: one call per head
        q = q.view(n, H, dq)
        q = torch.stack([F.batch_norm(q[:, h], None if s is None else s[0].to(f), None if s is None else s[1].to(f),
                                      None if gammas[h] is None else gammas[h].to(f),
                                      None if betas[h] is None else betas[h].to(f), s is None, 0.0, epss[h])
                         for h, s in enumerate(stats)], dim=1)
    q = q.view(n * H, dq)
    half = dq // 2
    # dense sub-scores, then the chosen columns: the backward is a GEMM for the keys
    s1 = (q[:, :half] @ k1.to(f).T).gather(1, (ids // K).view(n * H, -1))
    s2 = (q[:, half:] @ k2.to(f).T).gather(1, (ids % K).view(n * H, -1))
    return torch.softmax(s1 + s2, dim=-1).view(ids.shape)


class _GatePath(torch.autograd.Function):
    """The routing gates as one autograd node: forward the exact gates as float32, backward the
    derivative of _gate_values (ethos_gate_grads, which recomputes the queries from x).  wq and
    bq are the packed projections; `params` the tensors the gradients go to: weight and bias
    per head, both sub-key tables, the BatchNorms' weights, then their biases.  `stats`: None
    for batch statistics, or (means, variances) [H, d_query] at the time of the forward."""

    @staticmethod
    def forward(ctx, x, ids, gates, wq, bq, stats, eps, *params):
        ctx.save_for_backward(x, ids, wq, bq, *(stats or ()), *params)
        ctx.batch, ctx.eps = stats is None, eps
        return gates.to(torch.float32, copy=True)

    @staticmethod
    def backward(ctx, dg):
        x, ids, wq, bq = ctx.saved_tensors[:4]
        rest = ctx.saved_tensors[4:]
        stats, params = (None, rest) if ctx.batch else (rest[:2], rest[2:])
        H = wq.shape[0]
        head = (None,) * 6

        def split(ps):  # projection weights, biases, both sub-key tables, BatchNorm weights, biases
            return ps[0:2 * H:2], ps[1:2 * H:2], ps[2 * H:2 * H + 2], ps[2 * H + 2:3 * H + 2], ps[3 * H + 2:]

        if torch.is_grad_enabled():  # create_graph: the torch operations' own derivative
            # with respect to a view of each argument, which ends there: heads may share a
            # parameter, and x may itself come from one
            need = (ctx.needs_input_grad[0], *ctx.needs_input_grad[7:])
            ts = [t.view_as(t) if n else t for t, n in zip((x, *params), need)]
            w, b, (k1, k2), gamma, beta = split(ts[1:])
            g = _gate_values(ts[0], ids.long(), w, b, gamma, beta, k1, k2,
                             [None] * H if stats is None else list(zip(*stats)), [ctx.eps] * H)
            got = iter(torch.autograd.grad(g, [t for t, n in zip(ts, need) if n], dg, create_graph=True, allow_unused=True))
            out = [next(got) if n else None for n in need]
            return (out[0], *head, *out[1:])
        w, b, (k1, k2), gamma, beta = split(params)
        dx, dw, db, dgamma, dbeta, dk1, dk2 = hip.gate_grads(
            x, ids, dg.contiguous(), wq, bq, k1.detach(), k2.detach(), [t.detach() for t in gamma], [t.detach() for t in beta],
            stats and list(stats[0]), stats and list(stats[1]), ctx.eps, want_x=ctx.needs_input_grad[0],
            want_w=any(ctx.needs_input_grad[7:7 + 2 * H:2]))
        grads = [None] * (2 * H)
        if dw is not None:
            grads[0::2] = dw.unbind(0)
        grads[1::2] = db.unbind(0)
        return (dx, *head, *grads, dk1, dk2, *dgamma.unbind(0), *dbeta.unbind(0))


class _ExpertStages(torch.autograd.Function):
    """Expert generation, apply and scatter-back as one autograd node.

    Forward: the HIP generator and apply kernels, given the routing (gates, the sorted
    pair segments).  Backward: the derivative of the reference's per-pair expression
    (model.py:312-341), evaluated in float32 from the saved routing and generated rows.
    With A = W2[:d], B = W2[d:] (net.2.weight halves), C = W1 (net.0.weight), pair p of
    token t(p) using unique expert s(p):

        pre_s = z_s C^T,  h_s = gelu(pre_s),  v_s = h_s B^T,  xp_t = x_t A,
        c_p = h_s · xp_t,  a_p = gelu(c_p) g_p,  y_t = (1/H) Σ_p a_p v_s

    so with dY_t = dy_t / H:  da_p = dY_t · v_s = (dY_t B) · h_s;  dg_p = gelu(c_p) da_p;
    dc_p = g_p gelu'(c_p) da_p;  dxp_t = Σ_p dc_p h_s;  dh_s = Σ_p (dc_p xp_t + a_p dY_t B);
    dA = x^T dxp,  dB = dY^T hacc with hacc_t = Σ_p a_p h_s,  dx = dxp A^T;
    dpre = gelu'(pre) dh,  dC = dpre^T z,  dz = dpre C (added into the latent rows of the
    unique experts).  v rows are not needed.  One library call (ethos_expert_grads) computes
    all of it; outside its limits the per-pair terms, the token sums (hacc, dxp) and the expert
    sums (dh, summed over each expert's sorted pairs in a fixed order) come from
    ethos_expert_backward and the rest are torch GEMMs.  The backward is deterministic.
    Both execution orders (scatter of v rows, hidden-space reordering) compute this same
    function, so they share the backward.

    The gates enter as `gates_exact` (the values the forward uses) and `gate_path` (a
    float32 tensor of the same values carrying the router's graph), whose gradient is dg.
    """

    @staticmethod
    def forward(ctx, x, gate_path, latents_w, w1_w, w2_w, layer, gates_exact, seg):
        out, h = layer._expert_stages(x, gates_exact, seg)
        latents, w1, w2, _ = layer._generator_params(x.dtype, x.device)
        ctx.save_for_backward(x, gates_exact, h, seg["uniq"], seg["pair_slot"], seg["n_unique"], seg["perm"],
                              seg["sorted_slot"], seg["seg_off"], latents, w1, w2)
        ctx.heads, ctx.top_k = layer.num_heads, layer.top_k
        ctx.param_dtypes = (latents_w.dtype, w1_w.dtype, w2_w.dtype)
        return out

    @staticmethod
    def backward(ctx, dy):
        # v_s = h_s B^T never needs forming: dY_t . v_s = (dY_t B) . h_s, the dv_s B term of
        # dh_s is sum_p a_p (dY_t B), and dB = dv^T h = dY^T hacc with hacc_t = sum_p a_p h_s.
        x, gates, h, uniq, pair_slot, n_unique, perm, sorted_slot, seg_off, latents, w1, w2 = ctx.saved_tensors
        seg = {"pair_slot": pair_slot, "perm": perm, "sorted_slot": sorted_slot, "seg_off": seg_off, "uniq": uniq,
               "n_unique": n_unique}
        H, k = ctx.heads, ctx.top_k
        n, d = x.shape
        # one library call when every operand has the layer's dtype; torch operations for other
        # sizes and dtypes, and under create_graph
        if not torch.is_grad_enabled() and all(t == x.dtype for t in ctx.param_dtypes):
            dyc = dy.contiguous()
            if hip.expert_grads_supported(x, dyc, h, latents, w1, w2):
                dx, dg, dlat, dw1, dw2 = hip.expert_grads(x, dyc, h, latents, w1, w2, seg, gates, H, k)
                return dx, dg.view(gates.shape), dlat, dw1, dw2, None, None, None
        f = torch.float32
        U = int(n_unique.item())
        A, B, C = w2[:d].to(f), w2[d:].to(f), w1.to(f)
        xf = x.to(f)
        xp = xf @ A
        dY = dy.to(f) * (1.0 / H)
        dYB = dY @ B
        # per-pair terms, token sums and expert sums (ethos_expert_backward)
        dg, hacc, dxp, dh = hip.expert_backward(h, xp, dYB, seg, gates, H, k, U)
        dB = dY.T @ hacc
        dA = xf.T @ dxp
        dx = dxp @ A.T
        ids = uniq[:U].long()
        z = latents[ids].to(f)
        dpre = _gelu_grad(z @ C.T) * dh
        dC = dpre.T @ z
        dlat = torch.zeros(latents.shape, dtype=f, device=x.device)
        dlat.index_add_(0, ids, dpre @ C)
        lat_dt, w1_dt, w2_dt = ctx.param_dtypes
        return (dx.to(x.dtype), dg.view(gates.shape), dlat.to(lat_dt), dC.to(w1_dt),
                torch.cat([dA, dB], 0).to(w2_dt), None, None, None)


class ExpertGenerationNetwork(nn.Module):
    """latent [d_latent] -> [u ; v] [2 d_model] through Linear, GELU, Linear (no biases)."""

    def __init__(self, d_latent: int, d_model: int, d_intermediate: int):
        super().__init__()
        self.d_expert_params = 2 * d_model
        self.net = nn.Sequential(
            nn.Linear(d_latent, d_intermediate, bias=False),
            nn.GELU(),
            nn.Linear(d_intermediate, self.d_expert_params, bias=False),
        )

    def forward(self, latent_vector: torch.Tensor) -> torch.Tensor:
        return self.net(latent_vector)


class ProductKeyRouter(nn.Module):
    """Multi-head product-key router with per-head query BatchNorm and shared sub-keys."""

    def __init__(self, config):
        super().__init__()
        self.d_model = config.d_model
        self.num_experts = config.num_experts
        self.top_k = config.top_k
        self.d_query = config.d_query
        self.num_heads = config.num_routing_heads
        self.num_sub_keys = math.isqrt(self.num_experts)
        if self.num_sub_keys ** 2 != self.num_experts:
            raise AssertionError("num_experts must be a perfect square")
        self.query_projs = nn.ModuleList([nn.Linear(self.d_model, self.d_query) for _ in range(self.num_heads)])
        self.query_norms = nn.ModuleList([nn.BatchNorm1d(self.d_query) for _ in range(self.num_heads)])
        self.sub_keys_1 = nn.Embedding(self.num_sub_keys, self.d_query // 2)
        self.sub_keys_2 = nn.Embedding(self.num_sub_keys, self.d_query // 2)
        self._train_pass = 0
        self._kept_weights, self._kept_bn, self._kept_identity = _Kept(), _Kept(), _Kept()

    # -- parameter packing (cached until a parameter changes; made anew by every training pass) ---
    def _weight_sources(self) -> list:
        """The projection weights and sub-keys, read from the modules' parameter dicts directly
        (this runs on every call; nn.Module attribute lookup is slow)."""
        ts = []
        for m in self._modules["query_projs"]._modules.values():
            ts += (m._parameters["weight"], m._parameters["bias"])
        ts += (self._modules["sub_keys_1"]._parameters["weight"], self._modules["sub_keys_2"]._parameters["weight"])
        return ts

    def _bn_sources(self) -> list:
        ts = []
        for m in self._modules["query_norms"]._modules.values():
            ts += (m._parameters["weight"], m._parameters["bias"], m._buffers["running_mean"], m._buffers["running_var"])
        return ts

    def _batch_counts(self) -> list:
        return [m._buffers["num_batches_tracked"] for m in self._modules["query_norms"]._modules.values()]

    def _packed_sources(self) -> list:
        """The tensors the packed form is built from."""
        return self._weight_sources() + self._bn_sources()

    def _pack_mode(self) -> int:
        """Part of the packed forms' keys.  Evaluation (0) trusts the parameters' version counters.
        A training pass has its own number: between two of them an optimizer may write through
        `.data` or pointers, which moves no counter, so each packs anew, and so does the first
        evaluation after them."""
        return self._train_pass if any(m.training for m in self._modules["query_norms"]._modules.values()) else 0

    def _packed_weights(self, dtype: torch.dtype, device: torch.device, mode: int | None = None) -> _Weights:
        mode = self._pack_mode() if mode is None else mode
        key = (dtype, device, mode, tuple((t.data_ptr(), t._version) for t in self._weight_sources() if t is not None))
        w = self._kept_weights.get(key)
        if w is None:
            with _packing():
                wq = torch.stack([m.weight.detach() for m in self.query_projs]).to(device=device, dtype=dtype).contiguous()
                bq = torch.stack([m.bias.detach() for m in self.query_projs]).to(device=device, dtype=dtype).contiguous()
                k1 = self.sub_keys_1.weight.detach().to(device=device, dtype=dtype).contiguous()
                k2 = self.sub_keys_2.weight.detach().to(device=device, dtype=dtype).contiguous()
                w = _Weights(wq, bq, k1, k2, hip.key_norm_bounds(k1, k2), hip.route_prepare_keys(k1, k2) if k1.is_cuda else None,
                             hip.query_proj_prepare(wq) if wq.is_cuda else None)
            self._kept_weights.put(key, w, w, mode > 0)
        return w

    # the last packed weights' prepared forms, and the identity affine of the training-mode projection
    _key_norms = property(lambda self: self._kept_weights.value.key_norms)
    _keys_prepared = property(lambda self: self._kept_weights.value.keys_prepared)
    _wq_prepared = property(lambda self: self._kept_weights.value.wq_prepared)
    _identity = property(lambda self: self._kept_identity.value)

    def _bn_coefficients(self, device: torch.device):
        """(alpha, beta) of the eval-mode BatchNorms, float32 [H, d_query] on the device."""
        ts = self._bn_sources()
        key = (device, tuple((t.data_ptr(), t._version) for t in ts if t is not None))
        bn = self._kept_bn.get(key)
        if bn is None:
            with _packing():
                norms, H = list(self.query_norms), self.num_heads
                one = ts[0].dtype if ts[0] is not None else None
                if (device.type == "cuda" and H <= hip.MAX_BN_HEADS and len({m.eps for m in norms}) == 1
                        and all(m.affine and m.track_running_stats for m in norms) and one in (torch.float32, torch.bfloat16)
                        and all(t is not None and t.dtype == one and t.device == device and t.is_contiguous() for t in ts)):
                    # on the device: the host evaluation below waits for four tensors of every head
                    bn = hip.bn_coefficients(*([m.detach() for m in ts[i::4]] for i in range(4)), norms[0].eps, self.d_query,
                                             one, device)
                else:
                    ab = [_bn_eval_coefficients(m, self.d_query) for m in norms]
                    bn = tuple(torch.from_numpy(np.stack(c)).contiguous().to(device) for c in zip(*ab))
            self._kept_bn.put(key, bn, bn)
        return bn

    def _packed(self, dtype: torch.dtype, device: torch.device):
        """What an evaluation reads: the packed weights and the BatchNorm coefficients."""
        return self._packed_weights(dtype, device, 0)[:4] + tuple(self._bn_coefficients(device))

    def _bn_uses_batch_stats(self) -> bool:
        return any(m.training or not m.track_running_stats for m in self._modules["query_norms"]._modules.values())

    def _bn_one_call(self, x_flat: torch.Tensor) -> bool:
        """Whether the heads' training-mode BatchNorms run as one library call: all of them on
        batch statistics with one eps and momentum, affine, in the layer's dtype on its device,
        without gradients of their own, over at least two tokens (torch refuses fewer), and with
        running statistics of their own (heads that share them update them one after the other)."""
        norms = list(self.query_norms)
        m0 = norms[0]
        ts = self._bn_sources()
        updated = sorted(t.data_ptr() for t in ts[2::4] + ts[3::4] if t is not None)
        ts = [t for t in ts if t is not None]
        return (x_flat.shape[0] > 1 and self.num_heads <= hip.MAX_BN_HEADS and not torch.is_grad_enabled()
                and self.d_query % 4 == 0
                and all(m.affine and m.training and m.eps == m0.eps and m.momentum == m0.momentum
                        and m.track_running_stats == m0.track_running_stats
                        and (m.running_mean is not None) == m0.track_running_stats for m in norms)
                and all(t.dtype == x_flat.dtype and t.device == x_flat.device and t.is_contiguous() for t in ts)
                and all(q - p >= self.d_query * x_flat.element_size() for p, q in zip(updated, updated[1:])))

    def queries(self, x_flat: torch.Tensor, packed=None) -> torch.Tensor:
        """Per-head queries after BatchNorm, [n, H, d_query] (model.py:215-216).  `packed`:
        the result of _packed for x_flat's dtype and device, if the caller has it."""
        batch = self._bn_uses_batch_stats()
        if packed is not None:
            w = _Weights(*packed[:4], None, None, None)
            return self._batch_queries(x_flat, w) if batch else hip.query_proj(x_flat, w.wq, w.bq, *packed[4:])
        w = self._pass_weights(x_flat, batch)
        return self._batch_queries(x_flat, w) if batch else self._eval_queries(x_flat, w)

    def _pass_weights(self, x_flat: torch.Tensor, batch: bool) -> _Weights:
        """The packed weights of a pass that starts here."""
        if batch:
            self._train_pass += 1
        return self._packed_weights(x_flat.dtype, x_flat.device, None if batch else 0)

    def _eval_queries(self, x_flat: torch.Tensor, w: _Weights) -> torch.Tensor:
        return hip.query_proj(x_flat, w.wq, w.bq, *self._bn_coefficients(x_flat.device), prepared=w.wq_prepared)

    def _batch_queries(self, x_flat: torch.Tensor, w: _Weights) -> torch.Tensor:
        # Training-mode BatchNorm normalises with batch statistics and updates the
        # running stats: project with an identity affine, then normalise the projected queries.
        one = self._kept_identity.get(x_flat.device)
        if one is None:
            with _packing():
                ones = torch.ones((self.num_heads, self.d_query), dtype=torch.float32, device=x_flat.device)
                one = (ones, torch.zeros_like(ones))
            self._kept_identity.put(x_flat.device, one, one)
        q_lin = hip.query_proj(x_flat, w.wq, w.bq, *one, prepared=w.wq_prepared)
        if self._bn_one_call(x_flat):
            m0 = self.query_norms[0]
            ts, track = self._bn_sources(), m0.track_running_stats
            batch = None
            if q_lin.dtype == torch.bfloat16:
                # bf16 sub-scores are full of ties, so the last bit of a mean decides experts:
                # the statistics are torch's own, in the order in which batch_norm takes a head's,
                # and the layer chooses what it would choose there (float32 sums of another order
                # move about 1 row in 400 to another expert at 4,096 tokens, within rounding).
                # Several heads share a reduction where that leaves each column's order as it is:
                # up to 1,024 columns and 8,192 rows, or 4 Mi values, in whole blocks of 256
                # columns (4,096 tokens, 8 heads of 256: 428 us a head at a time, 120 in fours)
                H, dq, n = self.num_heads, self.d_query, x_flat.shape[0]
                cols = 1024 if n <= 8192 else dq
                while cols < 4096 and 2 * cols * n <= 1 << 22:
                    cols *= 2
                each = max(1, cols // dq) if dq % 256 == 0 else 1
                qf = q_lin.float().view(n, H * dq)
                pairs = [torch.var_mean(qf[:, h * dq:(h + each) * dq], 0, unbiased=False) for h in range(0, H, each)]
                batch = tuple([s for p in pairs for s in p[i].split(dq)] for i in (1, 0))
            out = hip.query_bn_train(q_lin, *([t.detach() for t in ts[i::4]] for i in range(2)),
                                     ts[2::4] if track else None, ts[3::4] if track else None,
                                     m0.momentum if m0.momentum is not None else 0.1, m0.eps, batch=batch)
            if track:
                torch._foreach_add_([m.num_batches_tracked for m in self.query_norms], 1)
                self._kept_bn.clear()  # the running statistics' version counters do not move
            return out
        outs = []
        for h, m in enumerate(self.query_norms):
            outs.append(F.batch_norm(q_lin[:, h], m.running_mean, m.running_var,
                                     m.weight if m.affine else None, m.bias if m.affine else None,
                                     m.training or not m.track_running_stats, m.momentum if m.momentum is not None else 0.1,
                                     m.eps))
            if m.training and m.track_running_stats:
                m.num_batches_tracked.add_(1)
        # batch_norm updated the running statistics in place without bumping their version
        # counters, so the cached eval-mode coefficients are stale
        if any(m.training and m.track_running_stats for m in self.query_norms):
            self._kept_bn.clear()
        return torch.stack(outs, dim=1).contiguous()

    def route(self, x_flat: torch.Tensor, mark=None):
        """(gates [n, H, k] x.dtype, expert ids [n, H, k] int32).  `mark(stage)`, if given,
        is called after each stage is enqueued (used to place timing events)."""
        batch = self._bn_uses_batch_stats()
        w = self._pass_weights(x_flat, batch)
        q = self._batch_queries(x_flat, w) if batch else self._eval_queries(x_flat, w)
        if mark is not None:
            mark("query_proj")
        out = hip.route_topk(q, w.k1, w.k2, self.top_k, key_norms=w.key_norms, prepared_keys=w.keys_prepared)
        if mark is not None:
            mark("route")
        return out

    def gate_path(self, x_flat: torch.Tensor, ids: torch.Tensor) -> torch.Tensor:
        """float32 gates [n, H, k] recomputed with torch operations from the chosen expert ids,
        carrying autograd to x, the query projections, the BatchNorm affine parameters and
        both sub-key tables as the reference's topk values and softmax do (model.py:215-234):
        g = softmax(q1 · K1[i1] + q2 · K2[i2]) with i1 = id // K, i2 = id % K.  BatchNorm uses
        the module's mode (batch statistics when training) without touching the running
        statistics, which the routing pass has already updated."""
        norms = list(self.query_norms)
        return _gate_values(x_flat, ids, [m.weight for m in self.query_projs], [m.bias for m in self.query_projs],
                            [m.weight if m.affine else None for m in norms], [m.bias if m.affine else None for m in norms],
                            self.sub_keys_1.weight, self.sub_keys_2.weight,
                            [None if m.training or not m.track_running_stats else (m.running_mean, m.running_var)
                             for m in norms], [m.eps for m in norms])

    def _gate_graph(self, x_flat: torch.Tensor, ids: torch.Tensor, gates: torch.Tensor) -> torch.Tensor:
        """A float32 [n, H, k] tensor of the gates carrying gate_path's graph (int32 ids): one
        autograd node whose backward is one library call where that takes the operands, else
        gate_path."""
        ws, bn, norms = self._weight_sources(), self._bn_sources(), list(self.query_norms)
        n, d = x_flat.shape
        batch = norms[0].training or not norms[0].track_running_stats
        plain = (hip.gate_grads_supported(n, d, self.num_heads, self.d_query, self.num_sub_keys, self.top_k)
                 and all((m.training or not m.track_running_stats) == batch and m.affine and m.eps == norms[0].eps for m in norms)
                 and all(t is not None and t.dtype == x_flat.dtype and t.device == x_flat.device and t.is_contiguous()
                         for t in ws + bn[0::4] + bn[1::4] + ([] if batch else bn[2::4] + bn[3::4]))
                 and x_flat.data_ptr() % 16 == 0 and ws[-1].data_ptr() % 16 == 0 and ws[-2].data_ptr() % 16 == 0
                 # forward-mode derivatives and tracing need the torch operations
                 and torch.autograd.forward_ad._current_level < 0 and not torch.compiler.is_compiling())
        if not plain:
            return self.gate_path(x_flat, ids.long())
        wq, bq = self._packed_weights(x_flat.dtype, x_flat.device)[:2]
        stats = None if batch else (torch.stack(bn[2::4]), torch.stack(bn[3::4]))
        return _GatePath.apply(x_flat, ids, gates, wq, bq, stats, norms[0].eps, *ws, *bn[0::4], *bn[1::4])

    def forward(self, x_flat: torch.Tensor):
        """(scores [n, H, k], expert ids [n, H, k] int64) as model.py:208-254.  With autograd
        enabled the scores carry the gradient of the reference's topk + softmax."""
        with torch.no_grad():
            gates, ids = self.route(_as_input(x_flat, 2))
        if _wants_grad(x_flat, self):
            g = self._gate_graph(x_flat, ids, gates)
            gates = gates + (g - g.detach()).to(gates.dtype)
        return gates, ids.long()


class EthosExpertLayer(nn.Module):
    """The ETHOS expert layer: product-key routing over num_experts generated experts,
    reordered execution by expert id, head-averaged weighted scatter-back."""

    def __init__(self, config, hidden_space: bool | None = None):
        super().__init__()
        self.d_model = config.d_model
        self.num_experts = config.num_experts
        self.top_k = config.top_k
        self.num_heads = config.num_routing_heads
        self.d_latent = config.d_latent
        self.d_hidden = config.d_intermediate_hypernet
        # Execution order of the expert stages: False (default) generates v_e = h_e W_v per
        # unique expert and scatters a_p v_e into the tokens (model.py:320-341, the layer's
        # rounding points); True is the paper's hidden-space reordering (Algorithm 1,
        # paper/ETHOS.pdf p.10): h_acc = sum_p a_p h_e per token, projected by W_v once.
        # Same function, different rounding points; no v rows.
        self.hidden_space = bool(getattr(config, "hidden_space", False) if hidden_space is None else hidden_space)
        self.expert_latents = nn.Embedding(config.num_experts, config.d_latent)
        self.generation_network = ExpertGenerationNetwork(config.d_latent, config.d_model,
                                                          config.d_intermediate_hypernet)
        self.router = ProductKeyRouter(config)
        self._kept_gen = _Kept()

    def _param_sources(self) -> list:
        """Every tensor a forward reads (router parameters and BatchNorm buffers, latents and
        both generator weights), looked up afresh through the modules' dicts, so that a
        replaced parameter object is seen too."""
        gen = self._modules["generation_network"]._modules["net"]._modules
        return self._modules["router"]._packed_sources() + [
            self._modules["expert_latents"]._parameters["weight"], gen["0"]._parameters["weight"],
            gen["2"]._parameters["weight"]]

    def packed_tensors(self) -> list:
        """The packed forms that the last evaluation read."""
        r = self.router
        return [t for kept in (r._kept_weights, r._kept_bn, self._kept_gen) for t in kept.value or () if t is not None]

    def _generator_params(self, dtype, device, mode: int | None = None):
        """(latents, W1, W2, W_u^T): the generator weights in the layer dtype on the device,
        and (bf16) the transpose of W2's first d_model rows, cached until a weight changes (as
        ProductKeyRouter._pack_mode says)."""
        ps = (self.expert_latents.weight, self.generation_network.net[0].weight, self.generation_network.net[2].weight)
        mode = self._modules["router"]._pack_mode() if mode is None else mode
        key = (dtype, device, mode, tuple((p.data_ptr(), p._version) for p in ps))
        gen = self._kept_gen.get(key)
        if gen is None:
            with _packing():
                if all(p.dtype == dtype and p.device == device and p.is_contiguous() for p in ps):
                    gen = tuple(p.detach() for p in ps)
                else:
                    gen = tuple(p.detach().to(device=device, dtype=dtype).contiguous() for p in ps)
                wut = gen[2][: self.d_model].t().contiguous() if dtype == torch.bfloat16 else None
            own = [t for t in gen if all(t.data_ptr() != p.data_ptr() for p in ps)]
            gen = self._kept_gen.put(key, gen + (wut,), own + [wut], mode > 0)
        return gen

    def _expert_stages(self, x_flat: torch.Tensor, gates: torch.Tensor, seg: dict, xp: torch.Tensor | None = None):
        """(out, h): generation over the unique experts, activations and scatter-back in the
        layer's execution order, as one library call (`xp`: the token projection, if already
        formed)."""
        latents, w1, w2, wut = self._generator_params(x_flat.dtype, x_flat.device)
        return hip.expert_forward(x_flat, latents, w1, w2, seg, gates, self.num_heads, self.top_k,
                                  hidden_space=self.hidden_space, wut=wut, xp=xp)

    def forward(self, x: torch.Tensor) -> torch.Tensor:
        if x.dim() != 3 or x.shape[-1] != self.d_model:
            raise RuntimeError(f"expected x of shape [batch, seq, {self.d_model}], got {tuple(x.shape)}")
        b, s, d = x.shape
        x_flat = _as_input(x, 3).view(-1, d)
        if x_flat.shape[0] == 0:
            return torch.zeros_like(x)
        return self.forward_flat(x_flat).view(b, s, d)

    def forward_flat(self, x_flat: torch.Tensor, mark=None, side_stream: torch.cuda.Stream | None = None) -> torch.Tensor:
        """The layer on [n_tok, d_model] rows (model.py:288-343), in eval mode one library call;
        with `mark` or `side_stream` (and in training mode) stage by stage.  `mark(stage)`, if given, is
        called after the query projection, the routing and the sort are enqueued on the
        current stream (the expert stages are one library call; hip.stage_events times the
        stages inside it).  `side_stream`: the token projection x W_u, which needs only x, runs
        there while the routing and the sort run on the current stream, which waits for it
        before the expert stages (worth its host cost under graph capture; see
        ethos_amd.graphs)."""
        if _wants_grad(x_flat, self):
            with torch.no_grad():
                gates, ids = self.router.route(x_flat)
                seg = hip.sort_segment(ids.view(-1), self.num_experts)
            g = self.router._gate_graph(x_flat, ids, gates)
            return _ExpertStages.apply(x_flat, g, self.expert_latents.weight, self.generation_network.net[0].weight,
                                       self.generation_network.net[2].weight, self, gates, seg)
        router = self._modules["router"]
        if mark is None and side_stream is None and x_flat.shape[0] > 0 and not router._bn_uses_batch_stats():
            with torch.no_grad():
                w = router._packed_weights(x_flat.dtype, x_flat.device, 0)
                packed = w[:4] + tuple(router._bn_coefficients(x_flat.device))
                gen = self._generator_params(x_flat.dtype, x_flat.device, 0)
                return hip.layer_forward(x_flat, packed, w.key_norms, w.keys_prepared, w.wq_prepared, gen,
                                         self.num_experts, self.top_k, self.hidden_space)
        with torch.no_grad():
            xp = None
            if side_stream is not None:
                cur = torch.cuda.current_stream(x_flat.device)
                _, _, w2, wut = self._generator_params(x_flat.dtype, x_flat.device)
                # allocated on the current stream, written on the side stream, which the
                # current stream waits for before any use
                xp = torch.empty((x_flat.shape[0], self.d_hidden), dtype=x_flat.dtype, device=x_flat.device)
                side_stream.wait_stream(cur)
                with torch.cuda.stream(side_stream):
                    hip.token_proj(x_flat, w2, wut, out=xp)
            gates, ids = self.router.route(x_flat, mark)
            if xp is None and ids.numel() <= hip.SMALL_SORT_MAX and x_flat.dtype == torch.bfloat16:
                # small batches: the token projection runs in the sort's launch, beside its
                # single workgroup
                _, _, w2, wut = self._generator_params(x_flat.dtype, x_flat.device)
                seg, xp = hip.sort_segment_token_proj(ids.view(-1), self.num_experts, x_flat, w2, wut)
            else:
                seg = hip.sort_segment(ids.view(-1), self.num_experts)
            if mark is not None:
                mark("sort_segment")
            if side_stream is not None:
                cur.wait_stream(side_stream)
            out, _ = self._expert_stages(x_flat, gates, seg, xp=xp)
        return out


def _wants_grad(x: torch.Tensor, module: nn.Module) -> bool:
    return torch.is_grad_enabled() and (x.requires_grad or any(p.requires_grad for p in module.parameters()))


def _as_input(x: torch.Tensor, dim: int) -> torch.Tensor:
    if x.dim() != dim:
        raise RuntimeError(f"expected a {dim}-d input, got shape {tuple(x.shape)}")
    if x.device.type != "cuda":
        raise RuntimeError(f"ETHOS expert layer runs on a HIP device only (input is on {x.device})")
    if not x.is_contiguous():
        # the reference's x.view(-1, d_model) (model.py:290) also requires a viewable input
        raise RuntimeError("input must be contiguous")
    return x


# The reference's two interchangeable layer classes (model.py:351-355).
SimplifiedHypernetMoE = EthosExpertLayer
FusedLowRankMoE_Reordered = EthosExpertLayer
