"""HdcMamba block and model on MI355X: the reference module surface over HIP kernels.

Drop-in for hdcmamba/model.py of N01N9/hdcmamba: the class and function names,
constructor signatures, parameter/buffer names and shapes, and the order in which
construction consumes the global RNG (so ``torch.manual_seed(s)`` followed by
construction yields the same weights) are those of the reference.  The forward of a
block runs, per layer:

    norm_conv (HIP)  ->  in_proj (the tiled HIP GEMM, or the fp32 one, at the sizes where it
    measured faster; else the library's)  ->  ssm (HIP) and slot state, scan and gate (HIP)
    writing one `combined` row buffer
    ->  bf16 without autograd: one HIP GEMM applying the row LayerNorm of `combined` in its
        epilogue (row statistics handed over by the ssm and gate kernels), out_proj and the
        residual add, in place on the residual stream;
        otherwise: row LayerNorm (HIP, in place) -> out_proj with the residual (fp32: the HIP
        GEMM at the sizes where it measured faster; else addmm)

A forward, a decode step and a training step of a block are one native call each
(csrc/native.cpp); the Python composition of the same kernels takes what that path leaves out
(HdcMamba9v3Block._native_ok).

Intended semantics are computed (see the oracle's docstring for the reference kernel
defects that are not reproduced).  Only GPU tensors are accepted; there is no CPU path.
"""
from __future__ import annotations

from dataclasses import dataclass

import torch
import torch.nn as nn
import torch.nn.functional as F
from torch.autograd import forward_ad
from torch.utils.checkpoint import checkpoint

from . import _ops

__all__ = ["HdcMamba9v3Block", "HdcMamba9v3Model", "FusedNormConv1dFunction",
           "fused_norm_conv1d_trainable", "RowLayerNormFunction", "layer_norm", "SlotSsmMixerFunction",
           "set_differentiable_mixer", "set_fused_out_proj", "set_fused_step_front", "BlockState"]


@dataclass
class BlockState:
    """What one block carries from a prefill into single-token steps.

    conv     [B,3,dm]     block-input rows t-3..t-1 (activation dtype; zero rows before the
                          sequence start, whose LayerNorm is the LayerNorm bias)
    h        [B,ds]       SSM state, fp32
    S_prev   [B,H,hd,hd]  slot state at the last chunk boundary, fp32
    S_intra  [B,H,hd,hd]  between the tokens of a chunk, the last token's effective slot
                          state (the chunk's own decayed sum plus gamma^c S_prev), fp32;
                          not read at a chunk start
    pos                   offset of the next token inside its chunk
    """
    conv: torch.Tensor
    h: torch.Tensor
    S_prev: torch.Tensor
    S_intra: torch.Tensor
    pos: int = 0


class FusedNormConv1dFunction(torch.autograd.Function):
    """LayerNorm + causal depthwise conv1d (width 4) on the HIP kernels.

    Same ``apply(x, norm_weight, norm_bias, conv_weight[D,4], conv_bias, eps)`` signature
    and backward outputs (dx and the four parameter gradients in x's dtype, None for eps)
    as hdcmamba/model.py:126-166.  The backward is the exact gradient of the forward,
    including the LayerNorm bias terms (also through the LayerNorm of the zero rows before
    the sequence start) that the reference's backward kernel leaves out, from fp32 row
    statistics.
    """

    @staticmethod
    def forward(ctx, x, norm_weight, norm_bias, conv_weight, conv_bias, eps):
        ctx.save_for_backward(x, norm_weight, norm_bias, conv_weight)
        ctx.eps = float(eps)
        if _ops.timer.active:
            return _ops.norm_conv(x, norm_weight, norm_bias, conv_weight, conv_bias, eps)
        return _ops.native().norm_conv_forward(x, norm_weight, norm_bias, conv_weight, conv_bias, ctx.eps, _ops._stream(x))

    @staticmethod
    def backward(ctx, grad_output):
        x, norm_weight, norm_bias, conv_weight = ctx.saved_tensors
        return (*_ops.native().norm_conv_backward(grad_output, x, norm_weight, norm_bias, conv_weight, ctx.eps,
                                                  _ops._stream(x)), None)


def fused_norm_conv1d_trainable(x, norm_layer, conv_layer):
    """hdcmamba/model.py:168-172: weights cast to x.dtype, conv weight squeezed to [D,4]."""
    return FusedNormConv1dFunction.apply(
        x, norm_layer.weight.to(x.dtype), norm_layer.bias.to(x.dtype),
        conv_layer.weight.squeeze(1).to(x.dtype), conv_layer.bias.to(x.dtype), norm_layer.eps)


class RowLayerNormFunction(torch.autograd.Function):
    """LayerNorm over the last dim on the HIP kernels, forward and backward, with the
    semantics of nn.LayerNorm / F.layer_norm (fp32 statistics, output in x's dtype).

    ``apply(x, weight, bias, eps)``; weight and bias may both be None (no affine).  The
    parameter gradients are summed over rows in fp32 in a fixed order and returned in the
    parameters' dtype.
    """

    @staticmethod
    def forward(ctx, x, weight, bias, eps):
        ctx.eps = float(eps)
        ctx.w_dtype = weight.dtype if weight is not None else None
        ctx.save_for_backward(x, weight)
        return _ops.layer_norm(x.contiguous(), weight, bias, eps)

    @staticmethod
    def backward(ctx, grad_out):
        x, weight = ctx.saved_tensors
        dx, dw, db = _ops.layer_norm_bwd(grad_out.to(x.dtype), x.contiguous(), weight, ctx.eps)
        if weight is None:
            return dx, None, None, None
        return dx, dw.to(ctx.w_dtype), db.to(ctx.w_dtype), None


def layer_norm(x, weight=None, bias=None, eps=1e-5):
    """Row LayerNorm on the HIP kernels; goes through RowLayerNormFunction when autograd
    needs its gradient (training the residual path, norm_final and the LM's norm_f)."""
    needs = torch.is_grad_enabled() and (x.requires_grad or any(
        t is not None and t.requires_grad for t in (weight, bias)))
    if needs:
        return RowLayerNormFunction.apply(x, weight, bias, eps)
    return _ops.layer_norm(x.contiguous(), weight, bias, eps)


class SlotSsmMixerFunction(torch.autograd.Function):
    """The block's SSM and slot memory + GroupNorm/gate on the HIP kernels, differentiable.

    ``apply(projs, A_log, gamma, gn_w, gn_b, d_state, d_model, num_heads, chunk)`` returns
    the ``combined`` rows [y_ssm | gated slot output] of the forward (model.py:345-380).
    The backward (no counterpart in the reference, whose kernels have no autograd) returns
    the gradients of projs, A_log and the GroupNorm parameters; gamma (the slot decay, a
    buffer refreshed from decay_log) is treated as a constant.  Slot part: two passes over the
    sequence (hdcm_slot_grad), the first from the segment states that the forward left; SSM
    part: the adjoint scan from the forward's y.
    """

    @staticmethod
    def forward(ctx, projs, A_log, gamma, gn_w, gn_b, ds, dm, H, C):
        _ops._on_gpu(projs)
        streams = _ops.native_streams(projs, projs.shape[1], ds, "auto")
        combined, ws = _ops.native().mixer_forward(projs, A_log, gamma, gn_w, gn_b, (ds, H, C), streams)
        ctx.save_for_backward(projs, A_log, gamma, gn_w, gn_b, combined, ws)
        ctx.dims = (ds, dm, H, C)
        ctx.seg_tiles = _ops.option_value("slot_seg_tiles")
        return combined

    @staticmethod
    def backward(ctx, dcomb):
        projs, A_log, gamma, gn_w, gn_b, combined, ws = ctx.saved_tensors
        ds, dm, H, C = ctx.dims
        if ctx.seg_tiles != _ops.option_value("slot_seg_tiles"):  # the states were cut into other segments
            ws = _ops.slot_workspace(projs, dm, H, C)
            _ops.slot_state(projs, 3 * ds, gamma, dm, H, C, ws)
        dprojs, dA, dgw, dgb = _ops.native().mixer_backward(dcomb, projs, A_log, gamma, gn_w, gn_b, combined, ws,
                                                            (ds, H, C), _ops._stream(projs))
        return dprojs, dA, None, dgw, dgb, None, None, None, None


class _PadRows(torch.autograd.Function):
    """x [B,L,dm] with ``pad`` zero rows in front of every sequence (hdcm_pad_rows_fwd)."""

    @staticmethod
    def forward(ctx, x, pad):
        ctx.pad = pad
        return _ops.native().pad_rows(x, pad, _ops._stream(x))

    @staticmethod
    def backward(ctx, g):
        return g[:, ctx.pad:, :], None


class BlockTrainFunction(torch.autograd.Function):
    """One block's training forward and its backward as two native calls: the forward keeps the
    block and its input only and the backward recomputes the body from the block's parameters of
    that moment, as the reference's checkpoint does (model.py:391-392).

    ``apply(block, x, pad, *params)`` on the chunk-aligned contiguous x [B, pad + L, dm] of which the
    output leaves out the first ``pad`` rows; params those of ``block._grad_params()``.  x is saved
    only where the backward needs the body (not where only x gets a gradient, which is dy, and the
    mixer is not differentiated).  A backward that is itself to be differentiated (create_graph)
    runs through the block's Python composition instead.
    """

    @staticmethod
    def forward(ctx, block, x, pad, *params):
        ctx.block, ctx.pad, ctx.mixer = block, pad, block.differentiable_mixer
        ctx.autocast = torch.is_autocast_enabled("cuda"), torch.get_autocast_dtype("cuda")
        ctx.body = ctx.mixer or ctx.needs_input_grad[3]
        ctx.dtype = x.dtype
        if ctx.body:
            ctx.save_for_backward(x)
        y = block._native_forward(x, train=True)
        # .data: a tensor of its own on that storage.  A view made in here could not be changed in place.
        return y[:, pad:, :].data if pad else y

    @staticmethod
    def backward(ctx, dy):
        block, pad = ctx.block, ctx.pad
        need = ctx.needs_input_grad
        if not ctx.body:
            return None, F.pad(dy.to(ctx.dtype), (0, 0, pad, 0)), None, None
        (x,) = ctx.saved_tensors
        params = block._grad_params(ctx.mixer)
        if torch.is_grad_enabled():
            with torch.enable_grad(), torch.amp.autocast("cuda", dtype=ctx.autocast[1], enabled=ctx.autocast[0]):
                y = block._inner_forward(x)[:, pad:, :]
            wanted = [t for t, n in zip((x, *params), (need[1], *need[3:])) if n]
            grads = iter(torch.autograd.grad(y, wanted, dy, create_graph=True, allow_unused=True))
            dx = next(grads) if need[1] else None
            return (None, dx, None, *(next(grads) if n else None for n in need[3:]))
        native = _ops.native()
        dyp = dy.to(ctx.dtype)
        dyp = native.pad_rows(dyp, pad, _ops._stream(x)) if pad else dyp.contiguous()
        if ctx.mixer:
            mask = [need[1], *need[3:10], False, *need[10:]]
        else:
            mask = [need[1], *[False] * 10, need[3]]
        g = native.block_backward(x, dyp, block._params(), block.norm.eps, (block.d_state, block.num_heads, block.chunk_size),
                                  block._native_streams(x), ctx.mixer, torch.cuda.tunable.is_enabled(), mask)
        if ctx.mixer:
            return (None, g[0], None, *g[1:8], *g[9:])
        return None, g[0], None, g[11]


class HdcMamba9v3Block(nn.Module):
    """SSM + slot-memory block (hdcmamba/model.py:300-394).

    ``forward(x[B,L,d_model]) -> (y[B,L,d_model], None)``.  L is left-padded with zero
    rows to a multiple of ``chunk_size`` and the pad is sliced off the output
    (model.py:388-389,394).

    As in the reference, backward reaches out_proj and the residual only: the SSM and slot
    kernels are constants for autograd.  With ``differentiable_mixer = True`` (an added
    option) the training forward runs them through SlotSsmMixerFunction instead, so
    in_proj, the LN+conv, A_log and the GroupNorm receive gradients too.

    ``fused_out_proj`` (added, on by default): without autograd and in bf16, the LayerNorm
    of `combined`, out_proj and the residual add run as one GEMM whose epilogue applies the
    LayerNorm (hdcm_rowln_gemm_fwd) at the shapes where that measured faster (see
    ``_fused_out``); otherwise as a row LayerNorm kernel and addmm.
    """

    # where the SSM's launch overlaps the slot kernels: "none" = a side stream joined before them,
    # "state" = beside the state pre-pass and scan, "after_state" = beside the scan and the gate
    # pass, "gate" = beside all three, "auto" = the current stream, before them.  The fork and join
    # of two streams cost more than the overlap gains once the host keeps the GPU busy: B=1
    # L=32768 d_model 1024 501-507 us per block with "auto" against 512-517 with "state", B=2 L=3001
    # d_model 768 125 against 136 us; in a recorded 24-layer forward the overlap lost as well (14.46
    # ms in sequence, 14.59 overlapped).  (The Python composition, whose launches are the slower
    # side, keeps "state" for "auto" outside graph capture.)
    ssm_overlap = "auto"
    # decode step: the LayerNorm + conv of the token and in_proj as one launch
    # (hdcm_norm_conv_in_proj_step_fwd: in_proj's weight stream starts while the conv rows are
    # computed; the same values as the two kernels) where in_proj runs on the wide skinny GEMM
    # (at least 2048 outputs, d_model <= 2048); set_fused_step_front switches it.
    fused_step_front = True

    def __init__(self, d_model=512, d_state=64, num_heads=8, chunk_size=256, differentiable_mixer=False,
                 fused_out_proj=True):
        super().__init__()
        self.differentiable_mixer = differentiable_mixer
        self.fused_out_proj = fused_out_proj
        self.d_model, self.d_state = d_model, d_state
        self.num_heads, self.chunk_size = num_heads, chunk_size
        self.head_dim = d_model // num_heads
        proj = 3 * d_state + 4 * d_model

        # Construction order fixes the RNG stream (model.py:306-327).
        self.norm = nn.LayerNorm(d_model)
        self.conv1d = nn.Conv1d(d_model, d_model, kernel_size=4, groups=d_model, padding=3, bias=True)
        with torch.no_grad():
            nn.init.normal_(self.conv1d.weight, std=0.02)
            self.conv1d.weight[:, 0, -1] += 1.0  # start close to the identity tap
            self.conv1d.bias.zero_()
        self.in_proj = nn.Linear(d_model, proj, bias=True)
        with torch.no_grad():
            lo, hi = 0.001, 0.1  # dt = softplus(bias) starts uniform in [lo, hi]
            dt0 = torch.rand(d_state) * (hi - lo) + lo
            self.in_proj.bias[:d_state] = torch.log(torch.exp(dt0) - 1.0)
            q0, gate0 = 3 * d_state, 3 * d_state + 3 * d_model
            nn.init.xavier_uniform_(self.in_proj.weight[q0:gate0])
            self.in_proj.bias[gate0:].fill_(1.0)
        self.A_log = nn.Parameter(torch.log(torch.linspace(0.99, 0.9999, d_state)))
        self.decay_log = nn.Parameter(torch.log(torch.full((num_heads,), 0.05)))
        self.out_proj = nn.Linear(d_state + d_model, d_model, bias=False)
        self.group_norm = nn.GroupNorm(num_heads, d_model)
        self.register_buffer("gamma_buf", torch.exp(-F.softplus(self.decay_log)))

    def _mixer(self, x, state=None, normalize=True, row_stats=None):
        """LN+conv, in_proj, SSM and slot+gate into one `combined` row buffer, then (with
        ``normalize``) its LayerNorm in place (model.py:338-382).  x: chunk-aligned [B,L,dm].
        With ``state``, the SSM and slot states after the last row are written into it.  With
        ``row_stats`` ([P, B*L, 2] fp32) the SSM and the gate also write each row's partial
        (sum, sum of squares): the SSM's 32-channel blocks first, then one part per head."""
        B, L, dm = x.shape
        ds, H, C = self.d_state, self.num_heads, self.chunk_size
        dtype = x.dtype
        x_conv = fused_norm_conv1d_trainable(x, self.norm, self.conv1d)
        w_in, b_in = self.in_proj.weight.to(dtype), self.in_proj.bias.to(dtype)
        # the SSM and slot kernels are constants for autograd, so projs needs no graph either
        if _ops.gemm_preferred(x_conv, w_in, b_in):
            projs = _ops.gemm(x_conv, w_in, b_in)
        elif _ops.gemm_f32_preferred(B * L, x_conv, w_in, b_in):
            projs = _ops.gemm_f32(x_conv.view(B * L, dm), w_in, b_in).view(B, L, -1)
        else:
            projs = F.linear(x_conv, w_in, b_in)
        combined = torch.empty(B, L, ds + dm, device=x.device, dtype=dtype)
        # The SSM and the slot kernels read projs and write disjoint columns of `combined`,
        # so the SSM may run on a side stream beside some of the slot kernels (ssm_overlap:
        # "state" = beside the state pre-pass and scan, "after_state" = beside the scan and
        # the gate pass, "gate" = beside all three, "none" = before them, the main stream
        # waiting for it; "auto" = "none" under graph capture, else "state").  The
        # join before the return orders every later use (and the allocator's reuse) of projs
        # and combined after the SSM.
        main = torch.cuda.current_stream(x.device)
        mode = self.ssm_overlap
        if mode == "auto":
            mode = "none" if torch.cuda.is_current_stream_capturing() else "state"
        side = _ops.side_stream(x.device)  # one stream per device: the scan's workspace is kept per stream

        def run_ssm():
            side.wait_stream(main)
            with torch.cuda.stream(side):
                _ops.ssm(projs, self.A_log, ds, combined[..., :ds], h_final=None if state is None else state.h,
                         row_stats=row_stats, stats_part=0)
            if mode == "none":
                main.wait_stream(side)

        gamma = self.gamma_buf.to(dtype)
        q_col = 3 * ds
        if self.head_dim > _ops.SLOT_MAX_HEAD_DIM:
            mode = "none"  # the scan first (run_ssm reads mode when called)
            run_ssm()
            self._wide_slot_gate(projs, combined, gamma, row_stats, state)
            if normalize:
                _ops.layer_norm(combined, eps=1e-5, out=combined)
            return combined.view(B * L, ds + dm)
        ws = _ops.slot_workspace(projs, dm, H, C)
        if mode != "after_state":
            run_ssm()
        _ops.slot_state(projs, q_col, gamma, dm, H, C, ws)
        if mode == "after_state":
            run_ssm()
        if mode == "state":
            main.wait_stream(side)
        _ops.slot_gate(projs, q_col, gamma, self.group_norm.weight, self.group_norm.bias, 1e-5, ws,
                       combined, ds, dm, H, C, S_final=None if state is None else state.S_prev,
                       row_stats=row_stats, stats_part=_ops.ssm_stats_parts(ds))
        if mode in ("gate", "after_state"):
            main.wait_stream(side)
        if normalize:
            _ops.layer_norm(combined, eps=1e-5, out=combined)
        return combined.view(B * L, ds + dm)

    def _wide_slot_gate(self, projs, combined, gamma, row_stats, state):
        """Slot memory + GroupNorm + gate for a head dim above the fused kernels' 128 (the
        reference pads any head dim, model.py:245-246,286): a head of hd = 2 hb columns runs as two
        sub-heads of hb through the plain slot pass (hdcm_slot_attend_fwd, the head's decay for
        both).  The scores split over the two key blocks, phi(q).phi(k) = sum_b phi(q_b).phi(k_b),
        so value block c of the output is attend(q_c, k_c, v_c) + attend(q_b, k_b, v_c), b != c: the
        first pass gives the equal-block terms, the second, after the two value halves of every
        head in projs are exchanged, the crossed ones (at the other half's columns); then the
        GroupNorm over all hd values of their sum and the gate (hdcm_gnorm_gate_fwd).  projs'
        value columns are left exchanged.  Forward only: hd a multiple of 32 up to 256, no state
        hand-off."""
        B, L, _ = projs.shape
        dm, ds, H, C = self.d_model, self.d_state, self.num_heads, self.chunk_size
        hd = dm // H
        if hd % 32 or hd > 2 * _ops.SLOT_MAX_HEAD_DIM:
            raise _ops.HdcmError(f"slot memory (head dim {hd})", -3)
        if state is not None:
            raise _ops.HdcmError(f"slot memory state hand-off (head dim {hd})", -3)
        q_col = 3 * ds
        g2 = gamma.repeat_interleave(2)
        ws = _ops.slot_workspace(projs, dm, 2 * H, C)
        y1 = torch.empty(B, L, dm, device=projs.device, dtype=projs.dtype)
        y2 = torch.empty_like(y1)
        _ops.slot_attend(projs, q_col, q_col + dm, q_col + 2 * dm, g2, dm, 2 * H, C, True, y1, 0, ws=ws)
        v = projs[..., q_col + 2 * dm:q_col + 3 * dm].unflatten(-1, (H, 2, hd // 2))
        v.copy_(v.flip(-2))
        _ops.slot_attend(projs, q_col, q_col + dm, q_col + 2 * dm, g2, dm, 2 * H, C, True, y2, 0, ws=ws)
        _ops.gnorm_gate(y1, y2, projs[..., q_col + 3 * dm:], self.group_norm.weight, self.group_norm.bias, 1e-5, H,
                        combined[..., ds:], row_stats=row_stats, stats_part=_ops.ssm_stats_parts(ds))

    # ------------------------------------------------------------------ native host path
    def _native_ok(self, x):
        """Whether the native host path (csrc/native.cpp) takes x: everything but empty inputs, heads
        wider than the fused slot kernels', launches being timed one by one, autocast to
        another dtype and forward-mode differentiation; the Python composition below takes the rest, with the same kernels."""
        return (x.dtype in _ops._DTYPES and self.head_dim <= _ops.SLOT_MAX_HEAD_DIM and x.numel() > 0
                and not _ops.timer.active and forward_ad._current_level < 0 and self.ssm_overlap in ("auto", "none", "state", "gate", "after_state")
                and (not torch.is_autocast_enabled("cuda") or torch.get_autocast_dtype("cuda") == x.dtype))

    def _params(self):
        """The parameters in the order the native host path takes them."""
        return [self.norm.weight, self.norm.bias, self.conv1d.weight, self.conv1d.bias, self.in_proj.weight,
                self.in_proj.bias, self.A_log, self.gamma_buf, self.group_norm.weight, self.group_norm.bias,
                self.out_proj.weight]

    def _grad_params(self, mixer=None):
        """Those that receive a gradient (``mixer``: with the differentiable mixer)."""
        if not (self.differentiable_mixer if mixer is None else mixer):
            return [self.out_proj.weight]
        p = self._params()
        return p[:7] + p[8:]  # gamma_buf is a constant

    def _native_streams(self, x):
        return _ops.native_streams(x, x.shape[1], self.d_state, self.ssm_overlap)

    def _native_forward(self, x, state=None, out=None, train=False):
        """The block body on chunk-aligned contiguous x without autograd (_inner_forward).  ``train``: as
        the composition runs with autograd, the row LayerNorm in a pass of its own before out_proj
        (two-pass variance, the weight as it is now: the folded form reads row sums kept until the
        weight's version changes, which a write through ``.data`` or a flat buffer does not do)."""
        fused = not train and self._fused_out(x)
        sums = self._out_weight_sums(x.dtype) if fused and _ops.rowln_stats_ok(x, self.d_model) else None
        return _ops.native().block_forward(
            x, self._params(), self.norm.eps, (self.d_state, self.num_heads, self.chunk_size), self._native_streams(x),
            out, fused, sums, torch.cuda.tunable.is_enabled(), None if state is None else state.h,
            None if state is None else state.S_prev)

    def _native_padded(self, x, pad, train=False):
        """_native_forward on x [B,L,dm] with ``pad`` zero rows in front, which the output leaves out."""
        if not pad:
            return self._native_forward(x.contiguous(), train=train)
        xp = _ops.native().pad_rows(x, pad, _ops._stream(x))
        return self._native_forward(xp, out=xp, train=train)[:, pad:, :]

    def _fused_out(self, x):
        """Whether out_proj runs as the GEMM with the LayerNorm folded in (bf16, no autograd).
        Measured: it pays on the decode step (<= 16 rows: the weight-streaming kernels) and
        up to ~1024 output tiles of 256 x 256 (the 32768-token d_model=1024 forward: 512);
        at the 131072-token d_model=2048 prefill (4096 tiles) hipBLASLt's out_proj plus the
        LayerNorm kernel is ~5 % faster than the tiled GEMM, so that shape keeps them."""
        if not (self.fused_out_proj and x.dtype == torch.bfloat16 and not torch.is_grad_enabled()
                and (self.d_state + self.d_model) % 8 == 0 and self.d_model % 4 == 0):
            return False
        rows = x.numel() // self.d_model
        tiles = -(-rows // 256) * -(-self.d_model // 256)
        return rows <= 16 or tiles <= 1024

    def _out_weight_sums(self, dtype):
        """Row sums of the out_proj weight as used (in ``dtype``), kept until the parameter changes (its
        storage or its version counter).  A refresh writes into the same buffer, so a recorded graph
        that reads it sees the new sums."""
        p = self.out_proj.weight
        key = (p.data_ptr(), p._version, dtype, p.device)
        if getattr(self, "_wsum_key", None) != key:
            old = getattr(self, "_wsum", None)
            if old is not None and old.device == p.device and old.numel() == p.shape[0]:
                _ops.row_sums(p.to(dtype), out=old)
            else:
                self._wsum = _ops.row_sums(p.to(dtype))
            self._wsum_key = key
        return self._wsum

    def refresh_derived_weights(self):
        """Bring the kept out_proj row sums up to date with the weight (a recorded forward
        graph calls this before each replay; it launches nothing when the weight is
        unchanged)."""
        if getattr(self, "_wsum_key", None) is None:
            return
        p = self.out_proj.weight
        if (p.data_ptr(), p._version) != self._wsum_key[:2]:
            self._out_weight_sums(self._wsum_key[2])

    def _fused_mixer_out(self, x, state, out=None):
        """x + out_proj(LN(combined)) for the fused path, x [B,L,dm]; into ``out`` (which may be
        x) when given.  With more rows than a decode step the SSM and gate kernels hand the
        row statistics to the GEMM (hdcm_rowln_gemm_stats_fwd); otherwise the GEMM takes them
        from its operands (hdcm_rowln_gemm_fwd)."""
        B, L, dm = x.shape
        w = self.out_proj.weight.to(x.dtype)
        x2 = x.reshape(B * L, dm)
        o2 = None if out is None else out.view(B * L, dm)
        if _ops.rowln_stats_ok(x2, dm):
            parts = _ops.ssm_stats_parts(self.d_state) + self.num_heads
            stats = torch.empty(parts, B * L, 2, device=x.device, dtype=torch.float32)
            c = self._mixer(x, state, normalize=False, row_stats=stats)
            y = _ops.rowln_gemm_stats(c, w, self._out_weight_sums(w.dtype), stats, x2, out=o2)
        else:
            c = self._mixer(x, state, normalize=False)
            y = _ops.rowln_gemm(c, w, x2, out=o2)
        return y.view(B, L, dm)

    def _differentiable_mixer(self, x):
        """_mixer with autograd through every stage (differentiable_mixer)."""
        B, L, dm = x.shape
        ds, H, C = self.d_state, self.num_heads, self.chunk_size
        dtype = x.dtype
        x_conv = fused_norm_conv1d_trainable(x, self.norm, self.conv1d)
        projs = F.linear(x_conv, self.in_proj.weight.to(dtype), self.in_proj.bias.to(dtype))
        # gamma is a constant here (the buffer may carry its construction graph, as in the
        # reference's register_buffer of exp(-softplus(decay_log)))
        combined = SlotSsmMixerFunction.apply(projs, self.A_log.to(dtype), self.gamma_buf.detach().to(dtype),
                                              self.group_norm.weight.to(dtype), self.group_norm.bias.to(dtype),
                                              ds, dm, H, C)
        return layer_norm(combined, eps=1e-5).view(B * L, ds + dm)

    def _inner_forward(self, x, state=None):
        """Block body on a chunk-aligned [B,L,dm] input; returns x + out_proj(LN(combined))."""
        B, L, dm = x.shape
        if not torch.is_grad_enabled() and self._native_ok(x):
            return self._native_forward(x, state)
        if self._fused_out(x):
            return self._fused_mixer_out(x, state)
        if self.differentiable_mixer and state is None and torch.is_grad_enabled():
            if self.head_dim > _ops.SLOT_MAX_HEAD_DIM:
                raise _ops.HdcmError(f"differentiable slot memory (head dim {self.head_dim})", -3)
            c = self._differentiable_mixer(x)
        else:
            c = self._mixer(x, state)
        return self._out_proj(x.reshape(B * L, dm), c).view(B, L, dm)

    def _out_proj(self, x, c, out=None):
        """x + c @ out_proj.weight^T of rows x [M, dm], c [M, ds + dm], into ``out`` (which may be x) when given."""
        w = self.out_proj.weight.to(x.dtype)
        if not torch.is_grad_enabled() and forward_ad._current_level < 0 and _ops.gemm_f32_preferred(x.shape[0], c, w, x):
            return _ops.gemm_f32(c, w, res=x, out=out)
        return torch.addmm(x, c, w.t()) if out is None else out.addmm_(c, w.t())

    def _residual_step_(self, r, state=None):
        """In-place variant for a model-owned residual stream r [B,L,dm] (chunk-aligned):
        r += out_proj(LN(combined)), with the GEMM accumulating straight into r."""
        B, L, dm = r.shape
        if not torch.is_grad_enabled() and self._native_ok(r) and r.is_contiguous():
            return self._native_forward(r, state, out=r)
        if self._fused_out(r):
            self._fused_mixer_out(r, state, out=r)
            return r
        c = self._mixer(r, state)
        r2 = r.view(B * L, dm)
        self._out_proj(r2, c, out=r2)
        return r

    # ------------------------------------------------------------------ prefill / decode
    def new_state(self, batch, device, dtype):
        """The state before any token (what a prefill of an empty sequence leaves)."""
        dm, ds, H, hd = self.d_model, self.d_state, self.num_heads, self.head_dim
        return BlockState(conv=torch.zeros(batch, 3, dm, device=device, dtype=dtype),
                          h=torch.zeros(batch, ds, device=device),
                          S_prev=torch.zeros(batch, H, hd, hd, device=device),
                          S_intra=torch.zeros(batch, H, hd, hd, device=device), pos=0)

    def _prefill_state(self, xp):
        """The state a prefill over chunk-aligned xp fills in: its last three rows kept here, h and
        S_prev left to the kernels that write them."""
        B, L, _ = xp.shape
        if L < 3 or xp.numel() == 0:
            state = self.new_state(B, xp.device, xp.dtype)
            state.conv[:, 3 - L:].copy_(xp)
            return state
        H, hd = self.num_heads, self.head_dim
        f32 = dict(device=xp.device, dtype=torch.float32)
        return BlockState(conv=xp[:, L - 3:].clone(memory_format=torch.contiguous_format),
                          h=torch.empty(B, self.d_state, **f32), S_prev=torch.empty(B, H, hd, hd, **f32),
                          S_intra=torch.zeros(B, H, hd, hd, **f32), pos=0)

    def prefill(self, x):
        """Forward over x [B,L,dm] that also returns the BlockState after its last token.
        The padded length is a multiple of the chunk, so the next token starts a chunk."""
        _ops._on_gpu(x)
        B, L_in, _ = x.shape
        pad = (self.chunk_size - (L_in % self.chunk_size)) % self.chunk_size
        if pad and not torch.is_grad_enabled() and self._native_ok(x):
            xp = _ops.native().pad_rows(x, pad, _ops._stream(x))
        else:
            xp = F.pad(x, (0, 0, pad, 0)).contiguous() if pad else x.contiguous()
        state = self._prefill_state(xp.detach())
        y = self._inner_forward(xp, state)
        return y[:, pad:, :], state

    def step(self, x, state, pos_dev=None):
        """One token per batch row: x [B,dm] -> y [B,dm]; ``state`` advances in place.
        With ``pos_dev`` (int32 device scalar) the chunk offset is read on the device and
        state.pos is left to the caller (graph replay)."""
        _ops._on_gpu(x)
        dm, ds, H, C = self.d_model, self.d_state, self.num_heads, self.chunk_size
        if not torch.is_grad_enabled() and self._native_ok(x):
            w = self.in_proj.weight
            front = (self.fused_step_front and x.dtype == torch.bfloat16 and w.shape[0] >= 2048
                     and 1 <= x.shape[0] <= _ops.SKINNY_MAX_ROWS and dm % 32 == 0 and dm <= 2048)
            y = _ops.native().block_step(
                x, self._params(), self.norm.eps, (ds, H, C), state.conv, state.h, state.S_prev, state.S_intra, state.pos,
                pos_dev, front, self._fused_out(x), _ops.step_workspace(x.device) if front else None, _ops._stream(x))
            if pos_dev is None:
                state.pos = (state.pos + 1) % C
            return y
        B = x.shape[0]
        dtype = x.dtype
        w_in, b_in = self.in_proj.weight.to(dtype), self.in_proj.bias.to(dtype)
        conv_w = self.conv1d.weight.squeeze(1)
        if self.fused_step_front and w_in.shape[0] >= 2048 and _ops.norm_conv_in_proj_step_ok(x, w_in):
            _, projs = _ops.norm_conv_in_proj_step(x, self.norm.weight, self.norm.bias, conv_w, self.conv1d.bias,
                                                   self.norm.eps, state.conv, w_in, b_in)
        else:
            xc = _ops.norm_conv_step(x, self.norm.weight, self.norm.bias, conv_w, self.conv1d.bias, self.norm.eps,
                                     state.conv)
            # few rows: the weight-streaming skinny GEMM; otherwise the library GEMM
            projs = _ops.skinny_linear(xc, w_in, b_in) if _ops.skinny_ok(xc, w_in) else F.linear(xc, w_in, b_in)
        combined = torch.empty(B, ds + dm, device=x.device, dtype=dtype)
        _ops.mixer_step(projs, self.A_log, ds, 3 * ds, self.gamma_buf.to(dtype), self.group_norm.weight,
                        self.group_norm.bias, 1e-5, state.h, state.S_prev, state.S_intra, state.pos, C,
                        combined, dm, H, pos_dev=pos_dev)
        w_out = self.out_proj.weight.to(dtype)
        if self._fused_out(x):  # LayerNorm folded into the (skinny) out_proj GEMM
            y = _ops.rowln_gemm(combined, w_out, x)
        else:
            _ops.layer_norm(combined, eps=1e-5, out=combined)
            if _ops.skinny_ok(combined, w_out):
                y = _ops.skinny_linear(combined, w_out, residual=x)
            else:
                y = torch.addmm(x, combined, w_out.t())
        if pos_dev is None:
            state.pos = (state.pos + 1) % C
        return y

    def _refresh_gamma(self):
        """gamma_buf from decay_log, as the reference does at every training forward (model.py:390)."""
        d, g = self.decay_log, self.gamma_buf
        with torch.no_grad():
            if (d.dtype == g.dtype and d.dtype in _ops._DTYPES and d.is_cuda and g.device == d.device and d.is_contiguous()
                    and g.is_contiguous() and not torch.is_autocast_enabled("cuda")):
                _ops.native().refresh_gamma(d, g, _ops._stream(g))
            else:
                g.copy_(torch.exp(-F.softplus(d)))

    def forward(self, x):
        _ops._on_gpu(x)
        B, L_in, _ = x.shape
        pad = (self.chunk_size - (L_in % self.chunk_size)) % self.chunk_size
        if self.training:
            self._refresh_gamma()
        if self._native_ok(x):
            if not torch.is_grad_enabled():
                return self._native_padded(x, pad), None
            if self.training:
                params = self._grad_params()
                if x.requires_grad or any(p.requires_grad for p in params):
                    xp = _PadRows.apply(x, pad) if pad else x.contiguous()
                    return BlockTrainFunction.apply(self, xp, pad, *params), None
                with torch.no_grad():
                    return self._native_padded(x, pad, train=True), None
        if pad > 0:
            x = F.pad(x, (0, 0, pad, 0))
        if self.training:
            # the reference checkpoints the block body in training (model.py:391-392): only
            # x is kept for backward and the body runs again when the gradient is needed
            y = checkpoint(self._inner_forward, x.contiguous(), use_reentrant=False)
        else:
            y = self._inner_forward(x.contiguous())
        return y[:, pad:, :], None


class HdcMamba9v3Model(nn.Module):
    """Stack of blocks plus a final LayerNorm (hdcmamba/model.py:396-404).

    ``num_slots`` is accepted and unused, as in the reference.  ``chunk_size`` is an
    added keyword; its default 256 is the value the reference hard-codes.
    """

    def __init__(self, d_model, n_layers, d_state, num_slots, num_heads=8, chunk_size=256):
        super().__init__()
        self.layers = nn.ModuleList([
            HdcMamba9v3Block(d_model=d_model, d_state=d_state, num_heads=num_heads, chunk_size=chunk_size)
            for _ in range(n_layers)])
        self.norm_final = nn.LayerNorm(d_model)

    def forward(self, x):
        return self._forward(x, owned=False)

    def _forward(self, x, owned, then=None):
        """forward; with ``owned`` (x is a temporary of the caller's, e.g. the LM's embedding
        output) an inference forward whose rows need no padding updates x itself as the
        residual stream instead of a copy of it.  ``then`` (an nn.LayerNorm, the LM's norm_f)
        is applied after norm_final, in inference as one fused pass over the rows."""
        _ops._on_gpu(x)
        chunks = {layer.chunk_size for layer in self.layers}
        if torch.is_grad_enabled() or len(chunks) != 1 or self.training:
            for layer in self.layers:
                x, _ = layer(x)
        else:
            # Inference: one residual stream updated in place by every block.  Each block
            # of the reference left-pads its own input with zero rows (model.py:388-389), so
            # the pad rows are zeroed again before every block.
            (C,) = chunks
            B, L, dm = x.shape
            pad = (C - L % C) % C
            if owned and pad == 0 and x.is_contiguous():
                r = x
            else:
                r = torch.empty(B, L + pad, dm, device=x.device, dtype=x.dtype)
                r[:, pad:].copy_(x)
            for layer in self.layers:
                if pad:
                    r[:, :pad].zero_()
                layer._residual_step_(r)
            x = r[:, pad:]
            if then is not None and _ops.layer_norm2_ok(x):
                nf = self.norm_final
                return _ops.layer_norm2(x.contiguous(), nf.weight, nf.bias, nf.eps, then.weight, then.bias, then.eps)
        x = layer_norm(x, self.norm_final.weight, self.norm_final.bias, self.norm_final.eps)
        return x if then is None else layer_norm(x, then.weight, then.bias, then.eps)

    def prefill(self, x):
        """Forward over x [B,L,dm] (inference) that also returns every block's BlockState."""
        _ops._on_gpu(x)
        chunks = {layer.chunk_size for layer in self.layers}
        if len(chunks) != 1:
            raise RuntimeError("prefill needs one chunk size for all blocks")
        (C,) = chunks
        B, L, dm = x.shape
        pad = (C - L % C) % C
        r = torch.empty(B, L + pad, dm, device=x.device, dtype=x.dtype)
        r[:, pad:].copy_(x)
        states = []
        with torch.no_grad():
            for layer in self.layers:
                if pad:
                    r[:, :pad].zero_()
                st = layer._prefill_state(r)
                layer._residual_step_(r, st)
                states.append(st)
        y = _ops.layer_norm(r[:, pad:].contiguous(), self.norm_final.weight, self.norm_final.bias,
                            self.norm_final.eps)
        return y, states

    def step(self, x, states, pos_dev=None, then=None):
        """One token per batch row through every block and norm_final: x [B,dm] -> [B,dm].
        ``then`` (an nn.LayerNorm, the LM's norm_f) is applied after norm_final in the same
        pass (hdcm_rowln2_fwd, bit-identical to two LayerNorm launches)."""
        with torch.no_grad():
            for layer, st in zip(self.layers, states):
                x = layer.step(x, st, pos_dev)
        nf = self.norm_final
        if then is not None and _ops.layer_norm2_ok(x):
            return _ops.layer_norm2(x.contiguous(), nf.weight, nf.bias, nf.eps, then.weight, then.bias, then.eps)
        x = _ops.layer_norm(x, nf.weight, nf.bias, nf.eps)
        return x if then is None else _ops.layer_norm(x, then.weight, then.bias, then.eps)


def set_fused_out_proj(module, enabled=True):
    """Switch the folded LayerNorm + out_proj GEMM of every HdcMamba9v3Block inside
    ``module`` on or off; returns ``module``."""
    for m in module.modules():
        if isinstance(m, HdcMamba9v3Block):
            m.fused_out_proj = bool(enabled)
    return module


def set_fused_step_front(module, enabled=True):
    """Switch the one-launch LayerNorm + conv + in_proj of the decode step of every
    HdcMamba9v3Block inside ``module`` on or off; returns ``module``."""
    for m in module.modules():
        if isinstance(m, HdcMamba9v3Block):
            m.fused_step_front = bool(enabled)
    return module


def set_differentiable_mixer(module, enabled=True):
    """Switch every HdcMamba9v3Block inside ``module`` to (or back from) the differentiable
    mixer; returns ``module``."""
    for m in module.modules():
        if isinstance(m, HdcMamba9v3Block):
            m.differentiable_mixer = bool(enabled)
    return module
