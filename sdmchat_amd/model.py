"""OneSdmLM: the whole language model around the run-time SDM mixer (experiments/track4/sdmllm/
track4_onesdm_models.py:471-555).

A drop-in for the reference model: the same constructor, module names and parameter creation order, and the same
initialisation rule, so a reference state dict loads with ``strict=True``.  Per layer, ``x + mems[i](x, reset)`` runs
the HIP mixer (RunTimeSdm) and the per-token step is either ``x + SwiGLU(RMSNorm x)`` (dense GEMMs) or
``x + TrainedSdm(x)`` (the product-key table layer); then the final RMSNorm and the tied head ``h @ E^T``.  The RMSNorms
run on the RMSNorm kernel; the dense maps are hipBLASLt GEMMs through torch.  The reference's archive memory is a
separate subsystem and is not built here (archive=True raises).

Training: with autograd recording the mixers run their differentiable path (core.MixerFunction, backward on the HIP
kernels), the TrainedSdm layers theirs (core.TableSdmFunction, sdm_rt_table_backward) and the model's own norms the
reference's torch ops, so every arm (ffn="mlp", "sdm", "none") trains.
"""
import math

import torch
import torch.nn as nn
import torch.nn.functional as F

from . import core
from .runtime_sdm import RMSNorm, RunTimeSdm
from .trained_sdm import TrainedSdm


def _norm(x, norm):
    """RMSNorm with the reference's dtype rule: cast_in(x * rsqrt(mean x^2 + eps)) * w, the result in the promoted
    dtype of x and w (track4_sdmllm_models.py:69-71).  On the kernel for inference; with autograd recording, the
    reference's own differentiable ops (the kernel has no backward)."""
    if torch.is_grad_enabled() and (x.requires_grad or norm.w.requires_grad):
        return norm(x)
    return core.rms_norm(x, norm.w, norm.eps, out_dtype=torch.promote_types(x.dtype, norm.w.dtype))


class SwiGLU(nn.Module):
    """down(silu(gate x) * up x) (track4_sdmllm_models.py:89-97).  Inference runs gate and up as one GEMM on their
    stacked weights and silu(g) * u as one kernel (core.silu_mul, torch's roundings); with autograd recording, the
    reference's ops."""

    def __init__(self, d, f):
        super().__init__()
        self.gate = nn.Linear(d, f, bias=False)
        self.up = nn.Linear(d, f, bias=False)
        self.down = nn.Linear(f, d, bias=False)
        self._gu = None

    def _gate_up(self):
        """[gate; up] stacked, cached until either changes."""
        key = tuple((w.data_ptr(), w._version, w.dtype) for w in (self.gate.weight, self.up.weight))
        if self._gu is None or self._gu[0] != key:
            self._gu = (key, torch.cat([self.gate.weight.detach(), self.up.weight.detach()], 0))
        return self._gu[1]

    def forward(self, x):
        if (torch.is_grad_enabled() and (x.requires_grad or any(p.requires_grad for p in self.parameters()))) \
                or x.device.type != "cuda" or torch.is_autocast_enabled("cuda"):
            return self.down(F.silu(self.gate(x)) * self.up(x))
        return core.linear(core.silu_mul(core.linear(x, self._gate_up())), self.down.weight, self.down.bias)


def trained_sdm_params(d, n_sub, heads, d_a):
    """Parameter count of one TrainedSdm (track4_onesdm_models.py:459-462)."""
    return d + d * heads * d_a + heads * n_sub * d_a + heads * n_sub * n_sub * (d // heads) + heads + d * d


def matched_sdm_n_sub(d, mlp_f, heads, d_a):
    """The n_sub whose TrainedSdm weight count is closest to one SwiGLU(d, mlp_f) plus its RMSNorm (:465-468)."""
    target = 3 * d * mlp_f + d
    return min(range(2, 4097), key=lambda n: abs(trained_sdm_params(d, n, heads, d_a) - target))


class ModelDecodeState:
    """The decode state of B streams of a OneSdmLM: per layer the mixer's core.DecodeState (None where the mixer is
    disabled) and the number of tokens each stream has consumed.  Everything else in the model acts per token."""

    def __init__(self, layers, pos=0):
        self.layers = list(layers)
        self.pos = pos

    def nbytes(self):
        """Device bytes the state holds."""
        return sum(st.nbytes() for st in self.layers if st is not None)


def decode_state_bytes(model, T):
    """Bytes kept to continue decoding after T tokens (float32), excluding the weights (track4_onesdm_models.py:
    641-652): per layer with a mixer, each head's M locations of dh values plus one write count.  It does not grow
    with T.  (ModelDecodeState.nbytes adds the per-head scales and last-write slots this build also keeps.)"""
    if not isinstance(model, OneSdmLM):
        raise ValueError(f"decode_state_bytes: {type(model).__name__} is not a OneSdmLM")
    if not model.has_mem:
        return 0
    m = model.mems[0]
    return model.n_layers * m.h * m.M * (m.dh + 1) * 4


class OneSdmLM(nn.Module):
    """Embedding, layers of [x + RunTimeSdm(x); x + FFN(x)], final RMSNorm, tied (or separate) head."""

    kind = "onesdm"

    def __init__(self, V, d=256, layers=4, mlp_f=688, mem=True, heads=4, n_sub=32, d_a=32, k=16,
                 decays=(0.0, 0.8, 0.99, 1.0), learn_decay=False, write_gate=True, gate_bias=0.0, read_mode="mean",
                 out_norm=True, addr_scale=8.0, learn_scale=True, chunk=128, mem_in_grad=1.0, out_norm_eps=1e-2,
                 read_eps=1e-3, addr_bias=0.0, archive=False,
                 arc_layers=None, arc_d_c=64, arc_n_sub=16, arc_k=4, arc_slot_keep=4, arc_window=16, arc_n_fetch=4,
                 arc_weighting="soft", tie=True, ffn="mlp", sdm_n_sub=0, sdm_heads=4, sdm_d_a=0, sdm_k=32,
                 sdm_scale=8.0, sdm_learn_scale=True, reset_at_bos=False, bos_id=0, seed=0):
        super().__init__()
        if ffn not in ("mlp", "sdm", "none"):
            raise ValueError("ffn must be 'mlp', 'sdm' or 'none'")
        if archive:
            raise NotImplementedError("OneSdmLM: the archive memory is a separate subsystem, not built here")
        self.V, self.d, self.n_layers, self.mlp_f, self.tie = V, d, layers, mlp_f, tie
        self.reset_at_bos, self.bos_id = reset_at_bos, bos_id
        self.ffn = ffn
        self.has_mem, self.has_arc = mem, False
        self.emb = nn.Embedding(V, d)
        self.mems = nn.ModuleList([RunTimeSdm(d, heads, n_sub, d_a, k, tuple(decays), learn_decay, write_gate,
                                              gate_bias, read_mode, out_norm, addr_scale, learn_scale, chunk,
                                              read_eps=read_eps, mem_in_grad=mem_in_grad, out_norm_eps=out_norm_eps,
                                              addr_bias=addr_bias, seed=seed + 31 * i) for i in range(layers)])
        for m in self.mems:
            m.enabled = mem
        if ffn == "mlp":
            self.mnorms = nn.ModuleList([RMSNorm(d) for _ in range(layers)])
            self.mlps = nn.ModuleList([SwiGLU(d, mlp_f) for _ in range(layers)])
        elif ffn == "sdm":
            self.sdm_d_a = sdm_d_a or min(32, (d // sdm_heads) // 2 * 2)
            self.sdm_n_sub = sdm_n_sub or matched_sdm_n_sub(d, mlp_f, sdm_heads, self.sdm_d_a)
            self.sdms = nn.ModuleList([TrainedSdm(d, self.sdm_n_sub, sdm_heads, self.sdm_d_a, sdm_k, sdm_scale,
                                                  sdm_learn_scale, seed=seed + 53 * i) for i in range(layers)])
        self.nf = RMSNorm(d)
        if not tie:
            self.head = nn.Linear(d, V, bias=False)
        nn.init.normal_(self.emb.weight, std=0.02)
        for n, p in self.named_parameters():
            if p.dim() == 2 and "emb" not in n and "onorm_w" not in n and "addr_b" not in n:
                out_map = n.endswith("down.weight") or (n.startswith("sdms.") and n.endswith("wo.weight"))
                nn.init.normal_(p, std=0.02 / math.sqrt(2 * layers) if out_map else 0.02)
        for m in self.mems:
            m.reset_init()
        for s in getattr(self, "sdms", []):
            s.reset_init()

    def enfold(self, idx):
        return self.emb(idx)

    def project(self, h):
        if self.tie:
            return core.linear(h, self.emb.weight, as_matmul=True)   # h @ E^T
        return core.linear(h, self.head.weight, self.head.bias)

    def unfold(self, x):
        return self.project(_norm(x, self.nf))

    def _inference(self):
        return not (torch.is_grad_enabled() and any(p.requires_grad for p in self.parameters())) \
            and not torch.is_autocast_enabled("cuda")

    def _stages(self):
        """The model's per-layer stages in order, each (kind, layer index, its input norm's weight and eps)."""
        out = []
        for i in range(self.n_layers):
            m = self.mems[i]
            if m.enabled:
                out.append(("mem", i, m.norm))
            if self.ffn == "mlp":
                out.append(("mlp", i, self.mnorms[i]))
            elif self.ffn == "sdm":
                out.append(("sdm", i, self.sdms[i].norm))
        return out

    def _norm_dtype(self, kind, i, x):
        """The dtype a stage's input norm produces: the mixer's and TrainedSdm's compute dtype, or the RMSNorm
        module's promoted dtype (the SwiGLU norms and nf)."""
        if kind == "mem":
            return self.mems[i]._compute_dtype(x)
        if kind == "sdm":
            return self.sdms[i]._compute_dtype(x)
        norm = self.mnorms[i] if kind == "mlp" else self.nf
        return torch.promote_types(x.dtype, norm.w.dtype)

    def _run(self, x, apply, apply_res=None, y0=None):
        """Inference: the residual stream through every stage with each residual add fused into the next stage's
        input norm (core.add_rms_norm: one kernel for x = x + y and its RMSNorm, the same roundings as the add and
        the norm apart); in front of a TrainedSdm stage that takes it (a few tokens, TrainedSdm.residual_fits) the
        add and the norm run inside that stage's table step instead (TrainedSdm.forward_residual, the same bits), and
        in front of a mixer whose decode step takes it (apply_res given, RunTimeSdm.residual_fits) inside the
        mixer's projection map (RunTimeSdm.step_residual, the same bits).  apply(kind, i, x, hx) gives a stage's
        output, apply_res(kind, i, x, y) a mixer's (x + y, output).  y0: the first stage's output, already computed
        from x by the caller (RunTimeSdm.step_embed).  Returns nf(x)."""
        stages = self._stages()
        if not stages:
            return _norm(x, self.nf)
        kind, i, norm = stages[0]
        x = x.contiguous()   # the residual stream (enfold's fresh output), updated in place
        if y0 is None:
            hx = core.rms_norm(x, norm.w, norm.eps, out_dtype=self._norm_dtype(kind, i, x))
        pending = None       # the last stage's output, to be added in front of this (TrainedSdm or mixer) stage
        for n, (kind, i, norm) in enumerate(stages):
            if n == 0 and y0 is not None:
                y = y0
            elif pending is not None:
                x, y = self.sdms[i].forward_residual(x, pending) if kind == "sdm" else apply_res(kind, i, x, pending)
                pending = None
            else:
                y = apply(kind, i, x, hx)
            nxt = stages[n + 1] if n + 1 < len(stages) else ("nf", 0, self.nf)
            if y.dtype != x.dtype:   # a stage wider than the stream: the add promotes, as x + y does
                x = (x + y).contiguous()
                hx = core.rms_norm(x, nxt[2].w, nxt[2].eps, out_dtype=self._norm_dtype(nxt[0], nxt[1], x))
                continue
            y = y.contiguous()
            if nxt[0] == "sdm" and self.sdms[nxt[1]].residual_fits(x, y):
                pending = y
                continue
            if nxt[0] == "mem" and apply_res is not None and self.mems[nxt[1]].residual_fits(x, y):
                pending = y
                continue
            x, hx = core.add_rms_norm(x, y, nxt[2].w, nxt[2].eps, out_dtype=self._norm_dtype(nxt[0], nxt[1], x))
        return hx

    def residual(self, idx, sequential=False):
        """The residual stream after the last layer (track4_onesdm_models.py:534-548).  ``sequential`` selects the
        token recurrence, which the HIP mixer computes in one pass either way."""
        x = self.enfold(idx)
        reset = (idx == self.bos_id) if self.reset_at_bos else None
        for i in range(self.n_layers):
            m = self.mems[i]
            if m.enabled:
                x = x + (m.forward_sequential(x, reset) if sequential else m(x, reset))
            if self.ffn == "mlp":
                x = x + self.mlps[i](_norm(x, self.mnorms[i]))
            elif self.ffn == "sdm":
                x = x + self.sdms[i](x)
        return x

    def hidden(self, idx, sequential=False):
        """The final normalised state the tied head reads (logits = hidden @ E^T)."""
        if self._inference() and idx.is_cuda:
            reset = (idx == self.bos_id) if self.reset_at_bos else None

            def apply(kind, i, x, hx):
                if kind == "mem":
                    return self.mems[i](x, reset, hx=hx)
                if kind == "mlp":
                    return self.mlps[i](hx)
                return self.sdms[i](x, hx=hx)
            return self._run(self.enfold(idx), apply)
        return _norm(self.residual(idx, sequential), self.nf)

    def forward(self, idx, sequential=False):
        return self.project(self.hidden(idx, sequential))

    def memory_parameters(self):
        """Names of the memories' parameters (track4_onesdm_models.py:557-558): the mixers' (``mems.``); the
        reference also lists its archive's (``arcs.``), which this model does not build."""
        return {n for n, _ in self.named_parameters() if n.startswith("mems.") or n.startswith("arcs.")}

    def set_leak(self, on):
        """The reference self-test's causality control (track4_onesdm_models.py:560-564): sets every mixer's
        ``_leak``.  The HIP mixers compute only the causal recurrence, so a forward with the control on raises."""
        for m in self.mems:
            m._leak = on

    # -- decoding ----------------------------------------------------------------------------------------------------
    def decode_state(self, batch, device=None):
        """An empty decode state for ``batch`` streams."""
        return ModelDecodeState([m.decode_state(batch, device) if m.enabled else None for m in self.mems])

    def prefill(self, idx):
        """forward(idx) over a prompt, also returning the decode state after its last token: (logits [B, T, V],
        ModelDecodeState), so step() continues the streams (inference only)."""
        keep = [m.keep_state for m in self.mems]
        try:
            for m in self.mems:
                m.keep_state = True
            logits = self.forward(idx)
            layers = []
            for m in self.mems:
                if m.enabled:
                    mem, cnt = m.last_state
                    layers.append(core.DecodeState.from_state(mem, cnt, core.pick_pitch(m.k, m.n_sub)))
                else:
                    layers.append(None)
        finally:
            for m, k in zip(self.mems, keep):
                m.keep_state = k
        return logits, ModelDecodeState(layers, idx.shape[1])

    def step(self, idx_t, state):
        """One token for each of B streams: idx_t [B] int64 -> logits [B, V], the last position of
        forward(idx, sequential=True) (track4_onesdm_models.py:534-555), with every mixer's memory carried in
        ``state`` (a ModelDecodeState, updated in place).  Inference only."""
        reset = (idx_t == self.bos_id) if self.reset_at_bos else None

        def apply(kind, i, x, hx):
            if kind == "mem":
                return self.mems[i].step(x, state.layers[i], reset, hx=hx)
            if kind == "mlp":
                return self.mlps[i](hx)
            return self.sdms[i](x[:, None], hx=hx[:, None])[:, 0]   # per token

        def apply_res(kind, i, x, y):   # a mixer's step on x + y, the add and its norm in the projection map
            return self.mems[i].step_residual(x, y, state.layers[i], reset)
        stages = self._stages()
        first = None   # a first mixer's step on the embedded tokens, the gather and its norm in the projection map
        if (stages and stages[0][0] == "mem" and type(self).enfold is OneSdmLM.enfold
                and self.mems[stages[0][1]].embed_fits(idx_t, self.emb.weight)):
            first = self.mems[stages[0][1]].step_embed(idx_t, self.emb.weight, state.layers[stages[0][1]], reset)
        h = self._run(first[0] if first else self.enfold(idx_t), apply, apply_res, y0=first[1] if first else None)
        state.pos += 1
        return self.project(h)


class DecodeGraph:
    """OneSdmLM.step for a fixed set of B streams captured in a HIP graph: ``step(tokens)`` copies the tokens into
    the graph's input, replays it and returns the graph's logits tensor (overwritten by the next step).  ``steps``
    consecutive steps can be captured in one graph (``run(tokens [steps, B])``).  The state is the caller's
    ModelDecodeState, updated in place; capture first runs two steps on a scratch state of the same shapes, so that
    every workspace and parameter cache exists before capture and nothing allocates inside the graph."""

    def __init__(self, model, state, steps=1):
        dev = model.emb.weight.device
        B = next(st.mem.shape[0] for st in state.layers if st is not None)
        self.model, self.state, self.steps = model, state, steps
        self.tokens = torch.zeros(steps, B, dtype=torch.long, device=dev)
        with torch.no_grad():
            scratch = model.decode_state(B, dev)
            for _ in range(2):
                model.step(self.tokens[0], scratch)
            torch.cuda.synchronize(dev)
            self.graph = torch.cuda.CUDAGraph()
            with torch.cuda.graph(self.graph):
                outs = [model.step(self.tokens[t], state) for t in range(steps)]
                self.logits = torch.stack(outs) if steps > 1 else outs[0]
        state.pos -= steps   # capture ran no step

    def run(self, tokens):
        """tokens [steps, B] (or [B] for one step) -> logits [steps, B, V] (or [B, V])."""
        self.tokens.copy_(tokens.reshape(self.tokens.shape))
        self.graph.replay()
        self.state.pos += self.steps
        return self.logits

    step = run


class ForwardGraph:
    """OneSdmLM.forward for token batches of one shape [B, T] captured in a HIP graph (prefill at a fixed shape):
    ``run(idx)`` copies the tokens into the graph's input, replays it and returns the graph's logits tensor
    (overwritten by the next run).  Capture first runs the forward twice on the same shapes, so that every workspace
    and parameter cache exists before capture; replays launch the whole forward at once, without the host's
    per-kernel work between launches.  Inference only; the model's parameters must not be replaced while the graph
    is in use (in-place updates are seen by the replays)."""

    def __init__(self, model, B, T):
        dev = model.emb.weight.device
        self.model = model
        # varied tokens for the warm-up forwards: a batch of one repeated token makes every position of a chunk pick
        # the same locations, the mixer core's slowest input (it costs time, not correctness)
        V = model.emb.weight.shape[0]
        self.idx = torch.arange(B * T, device=dev).mul_(7919).remainder_(V).view(B, T)
        with torch.no_grad():
            for _ in range(2):
                model(self.idx)
            torch.cuda.synchronize(dev)
            self.graph = torch.cuda.CUDAGraph()
            with torch.cuda.graph(self.graph):
                self.logits = model(self.idx)

    def run(self, idx):
        """idx [B, T] int64 -> logits [B, T, V]."""
        self.idx.copy_(idx)
        self.graph.replay()
        return self.logits
