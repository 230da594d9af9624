"""Ternary FFN block of the benchmark configuration (BitNet-2B shape):
RMSNorm(d_model) -> gate & up ternary linears (d_model -> d_ff) -> relu(gate)^2 * up ->
ternary down linear (d_ff -> d_model).

It is the caller of the ternary linear that the reference's GatedFFN.forward is
(src/rotor/transformer.py:320-341: gate_proj/up_proj on the same input, elementwise
activation, down_proj), with the configuration's relu^2 activation and no sub-norm.

On the GPU the block never leaves the device.  One token (decode) is two launches when
d_model and d_ff are multiples of 64 and d_ff <= 8192:
  1. gate/up pair plan over a copy of gate and up interleaved in 32-row groups: RMSNorm +
     int8 quantiser in the prologue, relu^2(gate) * up in the epilogue (rt_plan_create_gate_up)
  2. down plan quantising that row in its prologue            (rt_plan_create_fused)
Otherwise, and for several tokens, four:
  1. RMSNorm fused with the per-token int8 quantiser          (rt_act_rmsnorm_quantize)
  2. gate and up in one GEMV/GEMM launch on the shared int8 x (rt_plan_create_act)
  3. relu^2(gate) * up fused with the quantiser               (rt_act_relu2_mul_quantize)
  4. down on the int8 activations                             (rt_linear_act_f32)
where, past 64 tokens and at those widths, 2 runs on the interleaved copy and writes
relu^2(gate) * up itself (rt_plan_create_act_gate_up), half the bytes 3 then reads and
quantises.  All give the same bits.  No call allocates device memory after the first forward at a
given token count (and, for one token, input buffer), so a forward can be captured in a
HIP graph.
"""
from __future__ import annotations

import numpy as np

from .transformer import RMSNorm, TernaryLinear


class TernaryFFNBlock:
    def __init__(self, d_model: int, d_ff: int, use_gpu: bool = True, eps: float = 1e-6, max_tokens: int = 64):
        self.d_model, self.d_ff, self.eps = d_model, d_ff, eps
        self.use_gpu = use_gpu
        self.max_tokens = max_tokens
        self.norm = RMSNorm(d_model, eps)
        self.gate_proj = TernaryLinear(d_model, d_ff, use_gpu)
        self.up_proj = TernaryLinear(d_model, d_ff, use_gpu)
        self.down_proj = TernaryLinear(d_ff, d_model, use_gpu)
        self.gpu = self.gate_proj.gpu
        self._state = {}   # token count -> (plan, g, u, y); u None: g is relu^2(gate) * up
        self._acts = None
        self._norm_w_dev = None
        self._gu = None      # (gate, up, their interleaved copy for one token and past 64, scales)
        self._pair = None    # (input pointer, gate/up plan, down plan, y)
        self._xin = None     # forward()'s device copy of its input
        self.pair_ok = d_model % 64 == 0 and d_ff % 64 == 0 and d_ff <= 8192

    def load(self, norm_weight, gate, up, down):
        """gate/up/down: (rotor bytes [out, ceil(in/4)], scale) each.  A load that is refused, or
        for which the device has no room, leaves the block as it was.  At the widths of the
        interleaved copy it is laid out here (4.4 MB a matrix of 6912 x 2560), whatever token
        counts follow, so that no forward waits for it."""
        norm = np.asarray(norm_weight, dtype=np.float32)
        projs = (self.gate_proj, self.up_proj, self.down_proj)
        packed = [p._checked(*w) for p, w in zip(projs, (gate, up, down))]
        weights, gu = (None, None, None), None
        if self.use_gpu:
            import torch

            if self.pair_ok:
                gate_up, gu = self._upload_pair(packed)
            else:
                gate_up = [self.gpu.upload(b, self.d_model, s) for b, s in packed[:2]]
            weights = (*gate_up, self.gpu.upload(packed[2][0], self.d_ff, packed[2][1]))
            norm_dev = torch.from_numpy(norm.copy()).to(self.gpu.device)
            acts = (self.gpu.activations(self.max_tokens, self.d_model),
                    self.gpu.activations(self.max_tokens, self.d_ff))
        # all of it is accepted
        self.norm.weight = norm
        for p, (b, s), w in zip(projs, packed, weights):
            p._set(b, s, w)
        self._state.clear()
        self._pair = None
        if self.use_gpu:
            self._gu = (*gate_up, *gu) if gu is not None else None
            self._norm_w_dev, self._acts = norm_dev, acts

    def _upload_pair(self, packed):
        """Gate's and up's weights, and (interleaved matrix, scales) as
        HIPTernaryOps.interleave_gate_up returns them, from one device copy of the bytes."""
        import torch

        D, F = self.d_model, self.d_ff
        halves = [torch.from_numpy(np.require(b, requirements="W")).to(self.gpu.device) for b, _ in packed[:2]]
        scales = tuple(s for _, s in packed[:2])
        weights = [self.gpu.upload_device(h, D, s) for h, s in zip(halves, scales)]
        gu = torch.stack([h.view(F // 32, 32, -1) for h in halves], dim=1).view(2 * F, -1)
        return weights, (self.gpu.upload_device(gu, D, 1.0), scales)

    def _gate_up(self):
        """(interleaved matrix, scales) of gate's and up's present weights: load's, or a new one
        where either projection has been loaded on its own since."""
        gate, up = self.gate_proj.gpu_packed_weights, self.up_proj.gpu_packed_weights
        if self._gu is None or self._gu[0] is not gate or self._gu[1] is not up:
            self._gu = (gate, up, *self.gpu.interleave_gate_up(gate, up))
        return self._gu[2:]

    def _buffers(self, M):
        st = self._state.get(M)
        if st is None:
            import torch

            dev = self.gpu.device
            g = torch.empty((M, self.d_ff), dtype=torch.float32, device=dev)
            y = torch.empty((M, self.d_model), dtype=torch.float32, device=dev)
            act_h = self._acts[0]
            u = None
            if M > 64 and self.pair_ok:
                w_gu, scales = self._gate_up()
                plan = self.gpu.plan_act_gate_up(w_gu, scales, act_h, M, g)
            else:
                u = torch.empty((M, self.d_ff), dtype=torch.float32, device=dev)
                plan = self.gpu.plan_act([self.gate_proj.gpu_packed_weights, self.up_proj.gpu_packed_weights],
                                         [act_h, act_h], M, [g, u])
            st = self._state[M] = (plan, g, u, y)
        return st

    def _pair_plans(self, x):
        """One token: the gate/up pair plan and the down plan.  Plans hold the input
        pointer, so they are rebuilt when x is another buffer."""
        if self._pair is None or self._pair[0] != x.data_ptr():
            import torch

            from . import _hip

            hip, dev = self.gpu, self.gpu.device
            w_gu, scales = self._gate_up()
            a = torch.empty(self.d_ff, dtype=torch.float32, device=dev)
            ssq = torch.empty(self.d_ff // 32, dtype=torch.float64, device=dev)
            y = torch.empty((1, self.d_model), dtype=torch.float32, device=dev)
            gu = hip.plan_gate_up(w_gu, scales, _hip.SRC_RMSNORM, x.reshape(-1), self._norm_w_dev, eps=self.eps,
                                  a=a, ssq=ssq)
            down = hip.plan_fused([self.down_proj.gpu_packed_weights], _hip.SRC_QUANT, a, ys=[y.reshape(-1)])
            self._pair = (x.data_ptr(), gu, down, y)
        return self._pair

    def launches(self, M: int) -> int:
        """Kernel launches of one forward over M tokens."""
        return 2 if M == 1 and self.pair_ok else 4

    def forward_device(self, x):
        """x: device tensor [M, d_model] fp32 -> device tensor [M, d_model] (reused buffer)."""
        M = x.shape[0]
        if M > self.max_tokens:
            raise ValueError(f"{M} tokens exceed max_tokens={self.max_tokens}")
        if M == 1 and self.pair_ok:
            if not x.is_contiguous():
                raise ValueError("x must be contiguous")
            _, gu, down, y = self._pair_plans(x)
            gu.run()
            down.run()
            return y
        plan, g, u, y = self._buffers(M)
        act_h, act_a = self._acts
        hip = self.gpu
        hip.act_rmsnorm_quantize(x, self._norm_w_dev, act_h, self.eps)
        act_h.tokens = M
        plan.gemv()
        if u is None:
            hip.act_quantize(g, act_a)
        else:
            hip.act_relu2_mul_quantize(g, u, act_a)
        hip.linear_act(self.down_proj.gpu_packed_weights, act_a, out=y)
        return y

    def forward(self, x):
        """x [..., d_model] (numpy or torch) -> same leading shape, d_model."""
        if self.use_gpu:
            import torch

            shape = tuple(x.shape)
            xt = x if isinstance(x, torch.Tensor) else torch.from_numpy(np.ascontiguousarray(x, np.float32))
            xt = xt.to(self.gpu.device, torch.float32).reshape(-1, self.d_model)
            if self._xin is None:
                self._xin = torch.empty((self.max_tokens, self.d_model), dtype=torch.float32, device=self.gpu.device)
            xin = self._xin[:xt.shape[0]]
            xin.copy_(xt)  # one input buffer, so the one-token plans are built once
            y = self.forward_device(xin).clone().reshape(shape)
            return y if isinstance(x, torch.Tensor) else y.cpu().numpy()
        h = self.norm.forward(np.asarray(x, np.float32))
        g = self.gate_proj.forward(h)
        u = self.up_proj.forward(h)
        a = np.maximum(g, 0) ** 2 * u
        return self.down_proj.forward(a.astype(np.float32))
