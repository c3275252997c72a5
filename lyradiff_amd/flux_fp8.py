"""The FP8 feed-forward halves of the reference's FLUX blocks, built from the quantized-linear kernels.

Two reference call sequences are covered; attention itself (QKV/rotary/flash attention) is not part of the
quantized-linear path and stays with the caller, who passes its output in.

  FluxAttnPostFP8Processor<T>::forward   (layers/flux_attn_post_processor/FluxAttnPostFP8Processor.cc:93-240)
      hidden = input + gate_msa * attn          invokeFusedGateAndResidual
      norm   = adaLN(hidden, scale_mlp, shift_mlp)   invokeLayerNormWithShiftAndScale
      q1     = e4m3(norm / s_in1)               invokeCudaD2DScaleCpyConvert
      inner  = gelu(q1 . W1^T + b1)             GemmWithResidualAndBias (GELU_BIAS epilogue)
      q2     = e4m3(inner / s_in2)              invokeCudaD2DScaleCpyConvert
      ff     = q2 . W2^T + b2                   GemmWithResidualAndBias
      out    = hidden + gate_mlp * ff           invokeFusedGateAndResidual
    Seven launches and five 16-bit intermediate tensors there; three launches here, and only `hidden` is written
    in 16 bits: (1) gate+residual+adaLN+cast, (2) GEMM whose epilogue emits q2 directly, (3) GEMM whose epilogue
    applies the gate and the residual.

  FluxSingleTransformerFP8Block<T>::forward, after the attention (layers/flux_single_transformer_block/
  FluxSingleTransformerFP8Block.cc:209-290)
      q1   = e4m3(norm_hidden / s_mlp)          invokeCudaD2DScaleCpyConvert
      mlp  = q1 . Wm^T + bm                     GemmWithResidualAndBias
      cat  = [attn, gelu(mlp)]                  invokeFusedCatAndGelu
      q2   = e4m3(cat / s_out)                  invokeCudaD2DScaleCpyConvert
      o    = q2 . Wo^T + bo                     GemmWithResidualAndBias
      out  = input + gate * o                   invokeFusedGateAndResidual
    Here: the mlp GEMM writes the codes of gelu(mlp) straight into the right-hand columns of q2, a strided cast
    fills the left-hand (attention) columns, and the output GEMM applies gate and residual in its epilogue.

`msa` tensors follow the reference's layout [n_chunks, B, D] (AdaFP8LayerNorm.cc:100-175): for the double block
chunks 2..5 are gate_msa, shift_mlp, scale_mlp, gate_mlp; for the single block chunk 2 is the gate.
"""
from __future__ import annotations

from dataclasses import dataclass
from typing import Union

import torch

from . import ops
from .weights import FP8Linear, _source, load_fp8_linear


@dataclass
class FluxAttnPostFP8Weights:
    gelu_proj: FP8Linear  # "net.0.proj": [4D, D]
    ff_linear: FP8Linear  # "net.2":      [D, 4D]


@dataclass
class FluxSingleMlpFP8Weights:
    proj_mlp: FP8Linear  # "proj_mlp": [mlp_scale*D, D]
    proj_out: FP8Linear  # "proj_out": [D, (mlp_scale+1)*D]


def load_flux_attn_post_fp8(src, prefix: str, dim: int, dtype=torch.bfloat16, device="cuda", keep_master: bool = False):
    """Keys prefix + {"net.0.proj", "net.2"} + {".weight", ".bias", "_input_scale"}
    (FluxAttnPostFP8ProcessorWeight.cc:70-89; the block passes prefix + "ff." / "ff_context.")."""
    return FluxAttnPostFP8Weights(load_fp8_linear(src, prefix, "net.0.proj", 4 * dim, dim, dtype, device, keep_master),
                                  load_fp8_linear(src, prefix, "net.2", dim, 4 * dim, dtype, device, keep_master))


def load_flux_single_mlp_fp8(src, prefix: str, dim: int, mlp_scale: int = 4, dtype=torch.bfloat16, device="cuda",
                             keep_master: bool = False):
    """Keys prefix + {"proj_mlp", "proj_out"} + {".weight", ".bias", "_input_scale"}
    (FluxSingleTransformerFP8BlockWeight.cc:94-121)."""
    return FluxSingleMlpFP8Weights(
        load_fp8_linear(src, prefix, "proj_mlp", mlp_scale * dim, dim, dtype, device, keep_master),
        load_fp8_linear(src, prefix, "proj_out", dim, (mlp_scale + 1) * dim, dtype, device, keep_master))


def load_ada_fp8_layernorm(src, prefix: str, dim: int, n_chunks: int, dtype=torch.bfloat16, device="cuda",
                           keep_master: bool = False) -> FP8Linear:
    """Keys prefix + "linear" + {".weight", ".bias", "_input_scale"}, weight [n_chunks*D, D]
    (AdaFP8LayerNormWeight.cc:36-92; the blocks pass prefix + "norm1." / "norm1_context." / "norm.")."""
    return load_fp8_linear(src, prefix, "linear", n_chunks * dim, dim, dtype, device, keep_master)


@dataclass
class AdaLinear16:
    """The 16-bit adaLN linear of the quant levels FP8_W8A8 and INT4_W4A4 (AdaLayerNormWeight, keys prefix +
    "linear.weight" / ".bias"; the blocks take this branch unless the level is ..._FULL,
    FluxTransformerFP8Block.cc:203-211); the _FULL levels hold an FP8Linear in its place (AdaFP8LayerNormWeight)."""
    weight: torch.Tensor  # T [n_chunks*D, D]
    bias: torch.Tensor    # T [n_chunks*D]


def load_ada_layernorm(src, prefix: str, dim: int, n_chunks: int, full: bool, dtype=torch.bfloat16, device="cuda",
                       keep_master: bool = False) -> Union[FP8Linear, AdaLinear16]:
    """full: the level's adaLN linear is FP8 (keys with `_input_scale`); otherwise a plain 16-bit linear."""
    if full:
        return load_ada_fp8_layernorm(src, prefix, dim, n_chunks, dtype, device, keep_master)
    get = _source(src)
    return AdaLinear16(get(prefix + "linear.weight", (n_chunks * dim, dim), dtype).to(device),
                       get(prefix + "linear.bias", (n_chunks * dim,), dtype).to(device))


def _modulation_rows(temb: torch.Tensor, linear: Union[FP8Linear, AdaLinear16], dtype) -> torch.Tensor:
    if isinstance(linear, AdaLinear16):
        return ops.linear16(temb, linear.weight, linear.bias)
    flat = ops.fp8_linear_rows(temb, (linear.weight_rows32, linear.input_scale, linear.weight_scale, linear.bias)) if temb.dtype == dtype else None
    if flat is None:
        q = ops.fp8_scale_cast(temb, linear.input_scale)
        flat = ops.fp8_linear(q, linear.weight_rows32, linear.input_scale, linear.weight_scale, linear.bias, out_dtype=dtype)
    return flat


def ada_modulation(temb: torch.Tensor, linear: Union[FP8Linear, AdaLinear16], n_chunks: int, dtype, second=None):
    """msa [n_chunks, B, D] of the (already SiLU'd) time embedding temb [B, D]; with `second` (the other half's adaLN linear) a pair, in one
    launch where few rows let it.  16-bit linears are no quantized linears: a plain 16-bit matmul (AdaLayerNorm.cc)."""
    b, d = temb.shape
    lins = [linear] if second is None else [linear, second]
    flat = None
    if second is not None and all(isinstance(lin, AdaLinear16) for lin in lins):
        flat = ops.linear16_pair(temb, linear.weight, second.weight, linear.bias, second.bias)
    elif second is not None and temb.dtype == dtype and all(isinstance(lin, FP8Linear) for lin in lins):
        flat = ops.fp8_linear_rows(temb, *((lin.weight_rows32, lin.input_scale, lin.weight_scale, lin.bias) for lin in lins))
    if flat is None:
        flat = [_modulation_rows(temb, lin, dtype) for lin in lins]
    chunks = lambda f: f.view(b, n_chunks, d).transpose(0, 1).contiguous() if b > 1 else f.view(n_chunks, 1, d)  # invokeTranspose102
    return chunks(flat[0]) if second is None else (chunks(flat[0]), chunks(flat[1]))


def ada_fp8_layernorm(x: torch.Tensor, temb: torch.Tensor, linear: Union[FP8Linear, AdaLinear16], n_chunks: int, code_scales=(),
                      switch_scale: bool = False, eps: float = 1e-6, panels: bool = False, msa=None):
    """AdaFP8LayerNorm<T>::forward (layers/ada_layer_norm/AdaFP8LayerNorm.cc:93-205): msa = FP8 linear of the
    (already SiLU'd) time embedding, stored [n_chunks, B, D]; output = (1 + msa[1]) * LayerNorm(x) + msa[0]
    (msa[0]/msa[1] swapped with switch_scale).  x [B, S, D], temb [B, D]; msa given: that one instead.
    code_scales: () -> the 16-bit normalised tensor as the reference writes it; one or two fp32 [1] input scales ->
    the e4m3 codes for the FP8 linears that consume it instead (cast fused, no 16-bit tensor); with panels=True the codes
    are k-panels [D/64, B*S, 64] (ops.fp8_quant_panels) instead of [B, S, D].
    Returns (norm | codes | (codes_a, codes_b), msa)."""
    b, s, d = x.shape
    if msa is None:
        msa = ada_modulation(temb.reshape(b, d), linear, n_chunks, x.dtype)
    shift, scale = (msa[1], msa[0]) if switch_scale else (msa[0], msa[1])
    if len(code_scales) == 0:
        return ops.gate_residual_layernorm_mod(x, scale, shift, eps=eps), msa
    if len(code_scales) == 1:
        return ops.layernorm_mod_fp8(x, scale, shift, code_scales[0], eps, panels=panels), msa
    return ops.layernorm_mod_fp8_dual(x, scale, shift, code_scales[0], code_scales[1], eps, panels=panels), msa


def _gated_norm_codes(x, attn_output, msa, w: FluxAttnPostFP8Weights, eps: float):
    """The first launch of flux_attn_post_fp8: (codes for gelu_proj as k-panels, hidden)."""
    b, s, d = x.shape
    if tuple(msa.shape) != (6, b, d):
        raise ValueError("msa must be [6, B, D]")
    gate_msa, shift_mlp, scale_mlp = msa[2], msa[3], msa[4]
    # the two FP8 activations of the sequence travel as k-panels [K/64, B*S, 64] (whole cache lines for the GEMMs' transfers)
    return ops.gate_residual_layernorm_mod_fp8(attn_output, gate_msa, x, scale_mlp, shift_mlp, w.gelu_proj.input_scale, eps, panels=True)


def fp8_half(lin: FP8Linear, codes: torch.Tensor, **output) -> ops.FP8Half:
    return ops.FP8Half(codes, lin.weight_rows32, lin.input_scale, lin.weight_scale, lin.bias, **output)


def flux_attn_post_fp8(x: torch.Tensor, attn_output: torch.Tensor, msa: torch.Tensor, w: FluxAttnPostFP8Weights,
                       eps: float = 1e-6) -> torch.Tensor:
    """x, attn_output [B, S, D]; msa [6, B, D] -> output [B, S, D] in three launches."""
    b, s, d = x.shape
    q1, hidden = _gated_norm_codes(x, attn_output, msa, w, eps)
    q2 = ops.fp8_linear_codes_panels(q1, w.gelu_proj.weight_rows32, w.gelu_proj.input_scale, w.gelu_proj.weight_scale,
                                     w.gelu_proj.bias, w.ff_linear.input_scale, gelu=1, round_dtype=x.dtype)
    out = ops.fp8_linear_gated_panels(q2, w.ff_linear.weight_rows32, w.ff_linear.input_scale, w.ff_linear.weight_scale,
                                      w.ff_linear.bias, msa[5], hidden.view(b * s, d), rows_per_gate=s)
    return out.view(b, s, d)


def flux_attn_post_fp8_pair(x, attn_output, msa, w: FluxAttnPostFP8Weights, context, context_attn, context_msa, wc: FluxAttnPostFP8Weights,
                            eps: float = 1e-6):
    """flux_attn_post_fp8 of the image and of the text half of a double-stream block, their linears two to a launch."""
    q1, hidden = _gated_norm_codes(x, attn_output, msa, w, eps)
    c1, chidden = _gated_norm_codes(context, context_attn, context_msa, wc, eps)
    q2, c2 = ops.fp8_linear_pair(fp8_half(w.gelu_proj, q1, out_fp8_scale=w.ff_linear.input_scale),
                                 fp8_half(wc.gelu_proj, c1, out_fp8_scale=wc.ff_linear.input_scale), x.dtype, gelu=1)
    out, cout = ops.fp8_linear_pair(fp8_half(w.ff_linear, q2, gate=msa[5], residual=hidden, rows_per_gate=x.shape[1]),
                                    fp8_half(wc.ff_linear, c2, gate=context_msa[5], residual=chidden, rows_per_gate=context.shape[1]), x.dtype)
    return out.view(x.shape), cout.view(context.shape)


def flux_single_mlp_fp8(x: torch.Tensor, norm_hidden, attn_output: torch.Tensor, gate: torch.Tensor,
                        w: FluxSingleMlpFP8Weights, norm_in_panels: bool = False) -> torch.Tensor:
    """x, attn_output [B, S, D]; gate [B, D] (chunk 2 of the single block's msa) -> output [B, S, D].
    norm_hidden is either the 16-bit adaLN output [B, S, D] (cast here with proj_mlp's input scale) or its e4m3
    codes for proj_mlp: uint8 [B, S, D], or with norm_in_panels uint8 k-panels [D/64, B*S, 64] (the second output of
    ops.layernorm_mod_fp8_dual)."""
    b, s, d = x.shape
    m = b * s
    f = w.proj_mlp.weight_rows32.shape[0]
    if norm_hidden.dtype == torch.uint8 and not norm_in_panels:  # row-major codes from the caller: the row-major sequence
        q2 = torch.empty((m, d + f), dtype=torch.uint8, device=x.device)
        ops.fp8_scale_cast_into(attn_output.view(m, d), w.proj_out.input_scale, q2, 0)
        ops.fp8_linear_codes(norm_hidden.view(m, d), w.proj_mlp.weight_rows32, w.proj_mlp.input_scale, w.proj_mlp.weight_scale,
                             w.proj_mlp.bias, w.proj_out.input_scale, gelu=2, round_dtype=x.dtype, out=q2, col_offset=d)
        out = ops.fp8_linear_gated(q2, w.proj_out.weight_rows32, w.proj_out.input_scale, w.proj_out.weight_scale,
                                   w.proj_out.bias, gate, x.view(m, d), rows_per_gate=s)
        return out.view(b, s, d)
    # every FP8 activation as k-panels: the concatenated input of proj_out is [ (D + F)/64, M, 64 ], its two column blocks
    # (attention output, GELU of proj_mlp) are runs of whole panels
    q1 = norm_hidden if norm_hidden.dtype == torch.uint8 else ops.fp8_scale_cast_panels(norm_hidden.view(m, d), w.proj_mlp.input_scale)
    q2 = torch.empty(((d + f) // 64, m, 64), dtype=torch.uint8, device=x.device)
    ops.fp8_scale_cast_panels(attn_output.view(m, d), w.proj_out.input_scale, out=q2, col_offset=0)
    return _single_tail(x, q1, q2, gate, w)


def _single_tail(x, q1, q2, gate, w: FluxSingleMlpFP8Weights) -> torch.Tensor:
    """proj_mlp and proj_out: q1 the codes for proj_mlp, q2 those for proj_out whose first D columns (the attention output) are there."""
    b, s, d = x.shape
    ops.fp8_linear_codes_panels(q1, w.proj_mlp.weight_rows32, w.proj_mlp.input_scale, w.proj_mlp.weight_scale,
                                w.proj_mlp.bias, w.proj_out.input_scale, gelu=2, round_dtype=x.dtype, out=q2, col_offset=d)
    out = ops.fp8_linear_gated_panels(q2, w.proj_out.weight_rows32, w.proj_out.input_scale, w.proj_out.weight_scale,
                                      w.proj_out.bias, gate, x.view(b * s, d), rows_per_gate=s)
    return out.view(b, s, d)


# ---- whole blocks around a caller-supplied attention --------------------------------------------------------------------
# Everything the reference's FP8 blocks run through a quantized linear is here; `attention` is the caller's function
# for the part in between (q/k RMSNorm, rotary embedding, scaled-dot-product attention), which is not quantized.  The block ops pass a
# `core` instead (flux_ops.AttentionCore): this library's kernels for that part, whose output leaves the attention as codes.

@dataclass
class FluxSingleBlockFP8Weights:
    norm: Union[FP8Linear, AdaLinear16]  # prefix + "norm.linear"  [3D, D]
    to_qkv: FP8Linear    # prefix + "attn.to_qkv"  [3D, D]
    mlp: FluxSingleMlpFP8Weights


@dataclass
class FluxDoubleBlockFP8Weights:
    norm1: Union[FP8Linear, AdaLinear16]          # prefix + "norm1.linear"          [6D, D]
    norm1_context: Union[FP8Linear, AdaLinear16]  # prefix + "norm1_context.linear"  [6D, D]
    to_qkv: FP8Linear          # prefix + "attn.to_qkv"
    to_added_qkv: FP8Linear    # prefix + "attn.to_added_qkv"
    to_out: FP8Linear          # prefix + "attn.to_out.0"
    to_add_out: FP8Linear      # prefix + "attn.to_add_out"
    ff: FluxAttnPostFP8Weights          # prefix + "ff."
    ff_context: FluxAttnPostFP8Weights  # prefix + "ff_context."


def load_flux_single_block_fp8(src, prefix: str, dim: int, mlp_scale: int = 4, dtype=torch.bfloat16, device="cuda",
                               keep_master: bool = False, full: bool = True) -> FluxSingleBlockFP8Weights:
    """FluxSingleTransformerFP8BlockWeight::loadWeights (FluxSingleTransformerFP8BlockWeight.cc:94-121).
    full: quant level FP8_W8A8_FULL (FP8 adaLN linear); False: level FP8_W8A8 (16-bit adaLN linear)."""
    return FluxSingleBlockFP8Weights(load_ada_layernorm(src, prefix + "norm.", dim, 3, full, dtype, device, keep_master),
                                     load_fp8_linear(src, prefix + "attn.", "to_qkv", 3 * dim, dim, dtype, device, keep_master),
                                     load_flux_single_mlp_fp8(src, prefix, dim, mlp_scale, dtype, device, keep_master))


def load_flux_double_block_fp8(src, prefix: str, dim: int, dtype=torch.bfloat16, device="cuda",
                               keep_master: bool = False, full: bool = True) -> FluxDoubleBlockFP8Weights:
    """FluxTransformerFP8BlockWeight::loadWeights (FluxTransformerFP8BlockWeight.cc:78-91) and
    FluxAttentionFP8ProcessorWeight::loadWeights (FluxAttentionFP8ProcessorWeight.cc:113-138)."""
    lin = lambda name, n, k: load_fp8_linear(src, prefix + "attn.", name, n, k, dtype, device, keep_master)
    return FluxDoubleBlockFP8Weights(load_ada_layernorm(src, prefix + "norm1.", dim, 6, full, dtype, device, keep_master),
                                     load_ada_layernorm(src, prefix + "norm1_context.", dim, 6, full, dtype, device, keep_master),
                                     lin("to_qkv", 3 * dim, dim), lin("to_added_qkv", 3 * dim, dim), lin("to_out.0", dim, dim),
                                     lin("to_add_out", dim, dim),
                                     load_flux_attn_post_fp8(src, prefix + "ff.", dim, dtype, device, keep_master),
                                     load_flux_attn_post_fp8(src, prefix + "ff_context.", dim, dtype, device, keep_master))


def _linear_from_panels(lin: FP8Linear, panels: torch.Tensor, batch: int, dtype) -> torch.Tensor:
    """FP8 linear on codes in k-panels [K/64, B*S, 64] -> [B, S, N]."""
    y = ops.fp8_linear_panels(panels, lin.weight_rows32, lin.input_scale, lin.weight_scale, lin.bias, None, dtype)
    return y.view(batch, y.shape[0] // batch, y.shape[1])


def flux_single_block_fp8(x: torch.Tensor, temb: torch.Tensor, w: FluxSingleBlockFP8Weights, attention=None, core=None) -> torch.Tensor:
    """FluxSingleTransformerFP8Block<T>::forward (FluxSingleTransformerFP8Block.cc:163-291).  x [B, S, D], temb [B, D]
    (SiLU already applied); attention(qkv [B, S, 3D]) -> [B, S, D].  One adaLN read yields the codes for to_qkv and for
    proj_mlp; five launches besides the attention, four with a core."""
    b, s, d = x.shape
    (c_qkv, c_mlp), msa = ada_fp8_layernorm(x, temb, w.norm, 3, (w.to_qkv.input_scale, w.mlp.proj_mlp.input_scale), panels=True)
    qkv = _linear_from_panels(w.to_qkv, c_qkv, b, x.dtype)
    gate = msa[2].contiguous()
    if core is None:
        return flux_single_mlp_fp8(x, c_mlp, attention(qkv).contiguous(), gate, w.mlp, norm_in_panels=True)
    q2 = torch.empty((w.mlp.proj_out.weight_rows32.shape[1] // 64, b * s, 64), dtype=torch.uint8, device=x.device)
    core.codes(core.rotate(qkv), w.mlp.proj_out.input_scale, out=q2[: d // 64])
    return _single_tail(x, c_mlp, q2, gate, w.mlp)


def flux_double_block_fp8(x: torch.Tensor, context: torch.Tensor, temb: torch.Tensor, w: FluxDoubleBlockFP8Weights, attention=None, core=None):
    """FluxTransformerFP8Block<T>::forward (FluxTransformerFP8Block.cc:159-262) with FluxAttentionFP8Processor
    (FluxAttentionFP8Processor.cc:165-360).  attention(qkv [B, S, 3D], context_qkv [B, Sc, 3D]) -> (attn [B, S, D],
    context_attn [B, Sc, D]).  Returns (output, context_output)."""
    msa, cmsa = ada_modulation(temb.reshape(x.shape[0], x.shape[2]), w.norm1, 6, x.dtype, w.norm1_context)
    c, _ = ada_fp8_layernorm(x, temb, w.norm1, 6, (w.to_qkv.input_scale,), panels=True, msa=msa)
    cc, _ = ada_fp8_layernorm(context, temb, w.norm1_context, 6, (w.to_added_qkv.input_scale,), panels=True, msa=cmsa)
    parts = core.joint_qkv(x, context) if core is not None else None  # both halves side by side, where the batch lets them
    qkv, cqkv = ops.fp8_linear_pair(fp8_half(w.to_qkv, c, out=parts and parts[0]), fp8_half(w.to_added_qkv, cc, out=parts and parts[1]), x.dtype)
    if core is not None:
        cat = core.rotate(parts[2], context.shape[1]) if parts else core.rotate_two(qkv.view(*x.shape[:2], -1), cqkv.view(*context.shape[:2], -1))
        q, cq = core.codes(cat, w.to_out.input_scale, context.shape[1], w.to_add_out.input_scale)
    else:
        attn, cattn = attention(qkv.view(*x.shape[:2], -1), cqkv.view(*context.shape[:2], -1))
        q, cq = (ops.fp8_scale_cast_panels(t.contiguous().view(-1, t.shape[-1]), lin.input_scale)
                 for t, lin in ((attn, w.to_out), (cattn, w.to_add_out)))
    a_out, c_out = ops.fp8_linear_pair(fp8_half(w.to_out, q), fp8_half(w.to_add_out, cq), x.dtype)
    return flux_attn_post_fp8_pair(x, a_out.view(x.shape), msa, w.ff, context, c_out.view(context.shape), cmsa, w.ff_context)
