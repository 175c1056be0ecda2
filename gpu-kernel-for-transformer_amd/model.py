"""`UserOptimizedTransformer`: the drop-in causal pre-norm block stack on gfx950.

The module tree reproduces the reference's exactly -- ``layers.{i}.norm1``,
``layers.{i}.attention.{q,k,v,out}_proj``, ``layers.{i}.norm2``,
``layers.{i}.ffn_in``, ``layers.{i}.ffn_out``, ``final_norm``
(torch_transformer_benchmark.py:204-317) -- constructed in the same order, so
a strict `load_state_dict` from the reference's `BaselineTransformer` works
(torch_transformer_benchmark.py:1151-1161) and a seeded construction draws the
same nn.Linear initialisation.

`forward(x, valid_token_mask=None)` follows `_forward_cuda_fused_norm`
(torch_transformer_benchmark.py:1092-1148) with every device op a HIP kernel
from libxblock.so:

    n1 = LN(x)                                       xb_layernorm
    per layer:
      qkv = n1 . Wqkv^T + bqkv                       xb_linear        [M, 3D] fp16
      ctx = causal_attention(qkv)                    xb_attention     [M, D]  fp16
      a   = ctx . Wo^T + bo                          xb_linear        [M, D]  fp16
      x, n2 = x + a, LN2(x + a)                      xb_residual_layernorm
      h   = gelu_erf(n2 . W1^T + b1)                 xb_linear(GELU)  [M, F]  fp16
      f   = h . W2^T + b2                            xb_linear        [M, D]  fp16
      x, n1 = x + f, LN(x + f)  (next norm1, or final_norm in FP32 for the last layer)

The residual stream is FP32; GEMM operands are FP16 with FP32 accumulation,
the storage scheme of the reference's mixed-precision path.  There is no CPU
or PyTorch-op fallback: inputs that the HIP path cannot serve raise.

A padded `valid_token_mask` is handled as the reference's optimized path does
(torch_transformer_benchmark.py:497-513): padded tokens are masked as keys in
every layer's attention and their rows are zeroed only in the final
LayerNorm's output.  Valid rows therefore equal the baseline's, which also
zeroes padded rows after each attention and block (TTB:263-264, :290-291) --
padded rows reach valid ones only as keys, and those are masked.  Unlike the
reference (TTB:503-508) there is no sequence-length limit: the key mask is a
[B, S] byte vector read by the attention kernel, not a dense [S, S] mask.
`config.causal = False` runs the same kernels without the causal mask.
"""

from __future__ import annotations

import ctypes
import itertools
import operator
from typing import Dict, NamedTuple, Optional, Tuple

import torch
import torch.nn as nn

from . import _capi, kernels
from .config import (ShapeExecutionPlan, TransformerConfig, forward_working_set_bytes,
                     resolve_shape_execution_plan)

_LOG2E = 1.4426950408889634


class SelfAttentionParameters(nn.Module):
    """Parameter container with the reference's attention layout (TTB:207-220)."""

    def __init__(self, d_model: int, num_heads: int) -> None:
        super().__init__()
        if d_model % num_heads != 0:
            raise ValueError("d_model must be divisible by num_heads")
        self.d_model = d_model
        self.num_heads = num_heads
        self.head_dim = d_model // num_heads
        self.scale = self.head_dim**-0.5
        self.q_proj = nn.Linear(d_model, d_model, bias=True)
        self.k_proj = nn.Linear(d_model, d_model, bias=True)
        self.v_proj = nn.Linear(d_model, d_model, bias=True)
        self.out_proj = nn.Linear(d_model, d_model, bias=True)

    def forward(self, *args, **kwargs):  # pragma: no cover - explicit guard
        raise RuntimeError("run attention through UserOptimizedTransformer.forward")


class TransformerBlockParameters(nn.Module):
    """Parameter container with the reference's block layout (TTB:270-277)."""

    def __init__(self, d_model: int, num_heads: int, ffn_dim: int) -> None:
        super().__init__()
        self.norm1 = nn.LayerNorm(d_model)
        self.attention = SelfAttentionParameters(d_model, num_heads)
        self.norm2 = nn.LayerNorm(d_model)
        self.ffn_in = nn.Linear(d_model, ffn_dim)
        self.ffn_out = nn.Linear(ffn_dim, d_model)

    def forward(self, *args, **kwargs):  # pragma: no cover - explicit guard
        raise RuntimeError("run blocks through UserOptimizedTransformer.forward")


_DEVICE_OF, _EPS_OF, _SCALE_OF = map(operator.attrgetter, ("device", "eps", "scale"))
_VERSION_OF = operator.attrgetter("_version")  # raises RuntimeError on inference tensors, as _version does


def _tensor_version(tensor: torch.Tensor) -> Optional[int]:
    try:
        return tensor._version
    except RuntimeError:  # inference tensors expose no version counter
        return None


# Generation of the process's module trees: torch calls these global hooks
# whenever any nn.Module registers a parameter or a submodule by assignment,
# so a model's cached walk of its own tree (parameter list, LayerNorms) is
# redone only after some tree may have changed, not on every forward.  The
# walk itself (Module.parameters / modules) costs tens of microseconds, as
# much as a whole small forward.  No hook sees a module leave (`del
# model.layers[i]`, `pop`), enter by ModuleList.insert or by its parent's
# `_modules`: the walk's children are compared with the live ones as well.
_TREE_GENERATION = [0]


def _tree_changed(*_args) -> None:
    _TREE_GENERATION[0] += 1
    return None


nn.modules.module.register_module_parameter_registration_hook(_tree_changed)
nn.modules.module.register_module_module_registration_hook(_tree_changed)

_FLATTEN = itertools.chain.from_iterable


class _Tree(NamedTuple):
    """A walk of a model's modules.  The registries are the modules' own dicts, so looking
    through them again costs 1 to 2 us where walking the modules costs tens."""

    params: Tuple[nn.Parameter, ...]
    norms: Tuple[nn.LayerNorm, ...]
    attentions: Tuple[nn.Module, ...]
    generation: int
    children: Tuple[nn.Module, ...]
    child_registries: Tuple[dict, ...]      # `_modules` of every module that has children
    parameter_registries: Tuple[dict, ...]  # `_parameters` of every module that has some

    def live_children(self) -> Tuple[nn.Module, ...]:
        return tuple(_FLATTEN(map(dict.values, self.child_registries)))

    def live_parameters(self) -> Tuple[Optional[torch.Tensor], ...]:
        """What the modules hold now: torch.func.functional_call swaps tensors in without registering them."""
        return tuple(_FLATTEN(map(dict.values, self.parameter_registries)))


class _LayerWeights:
    """FP16 GEMM operands and FP32 biases of one block, as the kernels want them."""

    __slots__ = ("qkv_w", "qkv_b", "out_w", "out_b", "ffn_in_w", "ffn_in_b", "ffn_out_w", "ffn_out_b")

    def __init__(self, layer: TransformerBlockParameters) -> None:
        att = layer.attention
        with torch.no_grad():
            self.qkv_w = torch.cat((att.q_proj.weight, att.k_proj.weight, att.v_proj.weight), 0).to(torch.float16).contiguous()
            self.qkv_b = torch.cat((att.q_proj.bias, att.k_proj.bias, att.v_proj.bias), 0).float().contiguous()
            self.out_w = att.out_proj.weight.to(torch.float16).contiguous()
            self.out_b = att.out_proj.bias.float().contiguous()
            self.ffn_in_w = layer.ffn_in.weight.to(torch.float16).contiguous()
            self.ffn_in_b = layer.ffn_in.bias.float().contiguous()
            self.ffn_out_w = layer.ffn_out.weight.to(torch.float16).contiguous()
            self.ffn_out_b = layer.ffn_out.bias.float().contiguous()


class _RowBlockWeights:
    """One block's weights fragment-packed for xb_row_block, and its FP32 biases."""

    __slots__ = ("packed", "qkv_b", "out_b", "ffn_in_b", "ffn_out_b")

    def __init__(self, layer: TransformerBlockParameters) -> None:
        att = layer.attention
        linears = (att.q_proj, att.k_proj, att.v_proj, att.out_proj, layer.ffn_in, layer.ffn_out)
        with torch.no_grad():
            sizes = [lin.weight.numel() for lin in linears]
            self.packed = torch.empty(sum(sizes), device=att.q_proj.weight.device, dtype=torch.float16)
            for lin, part in zip(linears, self.packed.split(sizes)):
                kernels.pack_linear_fragments(lin.weight, out=part)
            self.qkv_b = torch.cat((att.q_proj.bias, att.k_proj.bias, att.v_proj.bias), 0).float().contiguous()
            self.out_b = att.out_proj.bias.float().contiguous()
            self.ffn_in_b = layer.ffn_in.bias.float().contiguous()
            self.ffn_out_b = layer.ffn_out.bias.float().contiguous()


class UserOptimizedTransformer(nn.Module):
    """Drop-in for the reference's UserOptimizedTransformer (TTB:320-1148), HIP-only."""

    def __init__(self, config: TransformerConfig) -> None:
        super().__init__()
        config.validate()
        self.config = config
        self.layers = nn.ModuleList(
            [
                TransformerBlockParameters(config.d_model, config.num_heads, config.ffn_dim)
                for _ in range(config.num_layers)
            ]
        )
        self.final_norm = nn.LayerNorm(config.d_model)
        # The gfx950 path computes GEMMs and attention in FP16 (FP32 accumulation,
        # FP32 residual stream); the reference reaches the same state through
        # enable_mixed_precision(torch.float16) (TTB:1750-1771).
        self._mixed_precision_dtype: Optional[torch.dtype] = torch.float16
        self._kv_cache_enabled = False
        self._kv_cache: Dict[int, Tuple[torch.Tensor, torch.Tensor]] = {}
        self._kv_cache_length = 0
        self._fused_stack_enabled = True
        self._large_batch_chunk_size = self.shape_execution_plan.batch_chunk_size
        self._strict_handoff_checks = False
        # Recorded for the reference's toggles (TTB:379-406); see their methods.
        self._triton_fused_norm_enabled = True
        self._triton_fused_ffn_enabled = True
        self._attention_fp16_accumulation_enabled = False
        self._walk()

    # What the forward derives from the module and rebuilds when it is missing.  A copy or a
    # saved file leaves it out (the descriptor's pointers are this process's and this model's),
    # and what a file saved with it holds is not taken over.
    _DERIVED = ("_native_stack_cache", "_weight_cache", "_fused_stack_cache", "_tree_cache", "_mask_cache",
                "_plans", "_plans_config")

    def __getstate__(self) -> dict:
        """The state that copy.deepcopy, pickle and torch.save take."""
        return {name: value for name, value in self.__dict__.items() if name not in self._DERIVED}

    def __setstate__(self, state: dict) -> None:
        super().__setstate__({name: value for name, value in state.items() if name not in self._DERIVED})

    # ----------------------------------------------------------------- toggles
    @property
    def shape_execution_plan(self) -> ShapeExecutionPlan:
        """The plan a forward of the config's own [batch_size, seq_len] input runs (TTB:364-367)."""
        cfg = self.config
        return self.execution_plan(cfg.batch_size, cfg.seq_len)

    def execution_plan(self, batch: int, seq_len: int, padded: bool = False, per_op: bool = False) -> ShapeExecutionPlan:
        """The kernels a forward of [batch, seq_len] runs (padded: a mask with a False), cached.

        The forward reads its kernel choices from here, so `describe()` of
        this plan names what runs.  Cached per shape and whole-stack
        eligibility (the enable_fused_stack toggle, LayerNorm eps and affine);
        per_op=True asks for the per-op sequence (KV-cached steps).
        """
        # Only a width-128 model can be eligible: the others don't pay for the question.
        eligible = not per_op and self.config.d_model == 128 and self._fused_stack_eligible()
        key = (int(batch), int(seq_len), bool(padded), eligible, bool(per_op),
               self._fused_stack_enabled)
        if self.__dict__.get("_plans_config") is not self.config:  # replaced: its plans with it
            self.__dict__["_plans_config"], self.__dict__["_plans"] = self.config, {}
        plans = self.__dict__["_plans"]
        plan = plans.get(key)
        if plan is None:
            plan = resolve_shape_execution_plan(self.config, batch, seq_len, masked=padded, fused_allowed=key[3],
                                                transposed_v_allowed=not per_op, row_block_allowed=key[5])
            plans[key] = plan
        return plan

    def activation_bytes(self, batch: int, seq_len: int) -> int:
        """Device bytes a forward of [batch, seq_len] keeps alive (input and output included)."""
        plan = self.execution_plan(batch, seq_len)
        return forward_working_set_bytes(self.config, batch, seq_len, fused=plan.fused)

    def enable_mixed_precision(self, dtype: Optional[torch.dtype] = torch.float16) -> None:
        """Select the compute dtype (TTB:369-377); the HIP path implements float16."""
        if dtype not in (None, torch.float16, torch.bfloat16):
            raise ValueError("mixed precision dtype must be float16 or bfloat16")
        if self._kv_cache_length:
            raise RuntimeError("reset the KV cache before changing precision")
        self._mixed_precision_dtype = dtype

    def enable_triton_fused_norm(self, enabled: bool = True) -> None:
        """Accepted for the reference's API (TTB:379-385); the gfx950 path has no Triton.

        Its residual-add + LayerNorm is always one HIP kernel (or part of the
        whole-stack kernel), so the flag is recorded and changes nothing.
        """
        self._triton_fused_norm_enabled = bool(enabled)

    def enable_triton_fused_ffn(self, enabled: bool = True) -> None:
        """Accepted for the reference's API (TTB:387-393); the FFN GEMM always carries its GELU epilogue."""
        self._triton_fused_ffn_enabled = bool(enabled)

    def enable_attention_fp16_accumulation(self, enabled: bool = True) -> None:
        """The reference's switch (TTB:395-406), same refusal for causal models.

        MFMA accumulates in FP32 at full rate, so on gfx950 the attention
        never accumulates in FP16; for a non-causal model the flag is recorded
        and changes nothing.
        """
        if enabled and self.config.causal:
            raise ValueError(
                "FP16 attention accumulation is disabled for causal models because it exceeds the accuracy tolerance")
        self._attention_fp16_accumulation_enabled = bool(enabled)

    def enable_fused_stack(self, enabled: bool = True) -> None:
        """Use the one-kernel whole-stack forward where its shape contract holds, and row blocks for narrow models.

        With it disabled every shape runs the per-op kernel sequence; the
        paths compute the same math (FP16 operands, FP32 accumulation).
        """
        self._fused_stack_enabled = bool(enabled)

    def enable_strict_handoff_checks(self, enabled: bool = True) -> None:
        """Synchronise after each split-form whole-stack launch and raise if a K/V hand-off failed.

        A failed hand-off (timed out, or published from another XCD) already
        turns the affected output rows into NaN;
        this debug mode turns it into a RuntimeError at the call (one host
        sync per forward).
        """
        self._strict_handoff_checks = bool(enabled)

    def enable_kv_cache(self, enabled: bool = True) -> None:
        """Incremental decoding over a per-layer FP16 KV cache, clearing any previous sequence (TTB:408-415).

        Each forward then appends its tokens (positions kv_cache_length ..)
        to the cache of capacity config.seq_len and attends causally over
        everything cached so far.
        """
        if enabled and not self.config.causal:
            raise ValueError("KV caching requires a causal Transformer")
        if enabled and self.training:
            raise RuntimeError("call eval() before enabling the KV cache")
        self._kv_cache_enabled = bool(enabled)
        self.reset_kv_cache()

    def reset_kv_cache(self) -> None:
        """Clear cached keys and values before starting a new sequence (TTB:417-420)."""
        self._kv_cache.clear()
        self._kv_cache_length = 0

    @property
    def kv_cache_length(self) -> int:
        return self._kv_cache_length

    # ------------------------------------------------------------ parameter caches
    def _layer_weights(self, index: int, form: type = _LayerWeights):
        """Packed FP16 weights of a layer in one form, rebuilt when any source parameter changes (TTB:524-641).

        Each form is kept by the parameters alone: a captured graph reads these buffers, so no
        setting (the row-block toggle, a LayerNorm's eps, the attention scale) may replace them.
        """
        layer = self.layers[index]
        params = list(layer.attention.parameters()) + list(layer.ffn_in.parameters()) + list(layer.ffn_out.parameters())
        key = tuple((p.data_ptr(), _tensor_version(p), p.device, p.dtype) for p in params)
        cache: Dict[Tuple[int, type], Tuple[tuple, object]] = self.__dict__.setdefault("_weight_cache", {})
        cached = cache.get((index, form))
        if cached is None or cached[0] != key or any(k[1] is None for k in key):
            cached = (key, form(layer))
            cache[(index, form)] = cached
        return cached[1]

    def _fits_config(self) -> bool:
        """Whether every parameter is what the native kernels index it as: of the config's
        sizes, all on one device, LayerNorms in contiguous float32."""
        d, f = self.config.d_model, self.config.ffn_dim
        square, vector = (d, d), (d,)
        tensors, norms = [], [self.final_norm]
        for layer in self.layers:
            parts = layer._modules  # read directly: nn.Module.__getattr__ made this a tenth of a first forward
            projections = parts["attention"]._modules
            norms += (parts["norm1"], parts["norm2"])
            for module, shape in ((projections["q_proj"], square), (projections["k_proj"], square),
                                  (projections["v_proj"], square), (projections["out_proj"], square),
                                  (parts["ffn_in"], (f, d)), (parts["ffn_out"], (d, f))):
                held = module._parameters
                weight, bias = held.get("weight"), held.get("bias")
                if weight is None or bias is None:
                    weight, bias = module.weight, module.bias  # parametrized, or missing
                if bias is None or weight.shape != shape or bias.shape != shape[:1]:
                    return False
                tensors += (weight, bias)
        for norm in norms:
            held = norm._parameters  # a parametrized one is made anew on each access: nothing to point at
            for p in (held.get("weight"), held.get("bias")):
                if p is None or p.shape != vector or p.dtype != torch.float32 or not p.is_contiguous():
                    return False
                tensors.append(p)
        return len(set(map(_DEVICE_OF, tensors))) == 1

    def _native_stack(self, row_block: bool) -> Optional[Tuple[_capi.XbStack, object, object, int]]:
        """(xb_stack, its xb_block array, the tensors they point into, their GPU), cached by parameter version.

        row_block: with fragment-packed weights for xb_row_block instead of
        the FP16 copies the GEMMs read.

        None when a parameter is missing or does not
        fit the config (_fits_config): the kernels would take its size from
        the config.  The wrappers, which take each size from the tensor
        itself, then run the forward or raise.  The descriptors are written
        once and only read afterwards, so forwards of several threads may
        share them.
        """
        tree = self._walk()
        params = tree.live_parameters()
        settings = (row_block, self.config, tuple(map(_EPS_OF, tree.norms)), tuple(map(_SCALE_OF, tree.attentions)))
        try:
            key = (tuple(map(_VERSION_OF, params)), tuple(map(torch.Tensor.data_ptr, params)), settings)
        except AttributeError:  # one is None (setting it calls no registration hook)
            return None
        except RuntimeError:  # inference-mode parameters have no version counter: never reuse
            key = None
        cached = self.__dict__.get("_native_stack_cache")
        if key is not None and cached is not None and cached[0] == key:
            return cached[1]
        if not self._fits_config():
            self.__dict__["_native_stack_cache"] = (key, None, params)
            return None
        cfg = self.config
        blocks = (_capi.XbBlock * len(self.layers))()
        form = _RowBlockWeights if row_block else _LayerWeights
        weights = [self._layer_weights(i, form) for i in range(len(self.layers))]
        for block, layer, w in zip(blocks, self.layers, weights):
            for name in w.__slots__:
                setattr(block, name, getattr(w, name).data_ptr())
            for which, norm in (("norm1", layer.norm1), ("norm2", layer.norm2)):
                setattr(block, which + "_g", norm.weight.data_ptr())
                setattr(block, which + "_b", norm.bias.data_ptr())
                setattr(block, which + "_eps", norm.eps)
                # The row blocks always apply it; asking costs two reads from the device.
                setattr(block, which + "_affine", int(row_block or self._layer_norm_uses_affine(norm)))
            block.scale = layer.attention.scale
        final = self.final_norm
        stack = _capi.XbStack(blocks=blocks, final_g=final.weight.data_ptr(), final_b=final.bias.data_ptr(),
                              final_eps=final.eps, final_affine=int(row_block or self._layer_norm_uses_affine(final)),
                              layers=len(self.layers), heads=cfg.num_heads, head_dim=cfg.head_dim,
                              ffn_dim=cfg.ffn_dim, causal=int(cfg.causal))
        value = (stack, blocks, weights, final.weight.get_device())
        # With the tensors that the key names: while it is compared against, nothing else can
        # come to lie at their addresses (tensors swapped in for one call are freed after it).
        self.__dict__["_native_stack_cache"] = (key, value, params)
        return value

    def _tree(self) -> Tuple[Tuple[nn.Parameter, ...], Tuple[nn.LayerNorm, ...]]:
        """(parameters, LayerNorm modules) of this model, as _walk found them."""
        tree = self._walk()
        return tree.params, tree.norms

    def _walk(self) -> _Tree:
        """This model's modules and parameters, re-walked after any registration or change of the modules."""
        cached = self.__dict__.get("_tree_cache")
        if (cached is None or cached.generation != _TREE_GENERATION[0]
                or cached.live_children() != cached.children):
            modules = tuple(self.modules())
            registries = tuple(m._modules for m in modules if m._modules)
            cached = _Tree(params=tuple(self.parameters()), norms=tuple(m for m in modules if isinstance(m, nn.LayerNorm)),
                           attentions=tuple(layer.attention for layer in self.layers), generation=_TREE_GENERATION[0],
                           children=tuple(_FLATTEN(map(dict.values, registries))), child_registries=registries,
                           parameter_registries=tuple(m._parameters for m in modules if m._parameters))
            self.__dict__["_tree_cache"] = cached
        return cached

    def _fused_stack_eligible(self) -> bool:
        """Conditions of the whole-stack kernel beyond the shape: the toggle, LayerNorm eps 1e-5 with affine."""
        if not self._fused_stack_enabled:
            return False
        # Parameters read from each module's registry directly: going through
        # nn.Module.__getattr__ for 18 of them cost microseconds per forward.
        for norm in self._walk().norms:
            registered = norm._parameters
            if norm.eps != 1e-5 or registered.get("weight") is None or registered.get("bias") is None:
                return False
        return True

    def _fused_stack_parameters(self) -> Tuple[torch.Tensor, torch.Tensor, int]:
        """Fragment-packed FP16 weights, FP32 bias/LayerNorm buffer and LayerNorm affine mask, cached by version."""
        params = self._walk().live_parameters()
        try:
            key = (tuple(map(_VERSION_OF, params)), tuple(map(torch.Tensor.data_ptr, params)))
        except AttributeError:  # a bias is None: the packing below raises for it
            key = None
        except RuntimeError:  # inference-mode parameters have no version counter: never reuse
            key = None
        cached = self.__dict__.get("_fused_stack_cache")
        if key is not None and cached is not None and cached[0] == key:
            return cached[1], cached[2], cached[3]
        weights, vectors = [], []
        with torch.no_grad():
            for layer in self.layers:
                att = layer.attention
                # softmax scale and log2(e) (the kernel exponentiates base 2) ride on Wq, bq
                q_scale = att.scale * _LOG2E
                for lin in (att.q_proj, att.k_proj, att.v_proj, att.out_proj, layer.ffn_in, layer.ffn_out):
                    weights.append(kernels.pack_linear_fragments(
                        lin.weight, scale=q_scale if lin is att.q_proj else 1.0))
                vectors.append(att.q_proj.bias.detach().float() * q_scale)
                for vec in (att.k_proj.bias, att.v_proj.bias, att.out_proj.bias,
                            layer.ffn_in.bias, layer.ffn_out.bias, layer.norm1.weight, layer.norm1.bias,
                            layer.norm2.weight, layer.norm2.bias):
                    vectors.append(vec.detach().float().reshape(-1))
            vectors += [self.final_norm.weight.detach().float(), self.final_norm.bias.detach().float()]
            wpack = torch.cat(weights).contiguous()
            ppack = torch.cat(vectors).contiguous()
        affine_mask = self._fused_affine_mask()
        self.__dict__["_fused_stack_cache"] = (key, wpack, ppack, affine_mask, params)  # held as in _native_stack
        return wpack, ppack, affine_mask

    def _fused_affine_mask(self) -> int:
        """Bit 2l / 2l+1: layer l's norm1 / norm2 has a non-identity affine (see xb_fused_forward_d128)."""
        mask = 0
        for index, layer in enumerate(self.layers[:31]):
            mask |= int(self._layer_norm_uses_affine(layer.norm1)) << (2 * index)
            mask |= int(self._layer_norm_uses_affine(layer.norm2)) << (2 * index + 1)
        return mask if len(self.layers) <= 31 else -1

    @staticmethod
    def _layer_norm_uses_affine(layer_norm: nn.LayerNorm) -> bool:
        """Whether gamma/beta differ from (1, 0), cached per version (TTB:568-596)."""
        weight, bias = layer_norm.weight, layer_norm.bias
        if weight is None or bias is None:
            return False
        versions = (_tensor_version(weight), _tensor_version(bias))
        if None in versions:
            return True
        key = (weight.data_ptr(), versions[0], bias.data_ptr(), versions[1])
        cached = getattr(layer_norm, "_xblock_affine_cache", None)
        if cached is None or cached[0] != key:
            with torch.no_grad():
                is_identity = bool(torch.all(weight == 1).item()) and bool(torch.all(bias == 0).item())
            cached = (key, not is_identity)
            layer_norm._xblock_affine_cache = cached
        return cached[1]

    def _single_launch_forward(self, x: torch.Tensor, valid_token_mask: Optional[torch.Tensor]) -> bool:
        """Whether forward(x, valid_token_mask) is exactly one kernel launch (the whole-stack kernel).

        Such a forward gains nothing from graph replay, which would only add
        the copy of the static output that every replay returns.  A mask with
        every token valid (the reference harness's timed input, TTB:1478-1491)
        runs the unmasked kernels, so it counts as no mask; one with padding
        is read as it is where its bytes are contiguous.
        """
        if not (not self._kv_cache_enabled and x.is_cuda and x.ndim == 3
                and x.dtype == torch.float32 and x.is_contiguous() and x.shape[-1] == self.config.d_model):
            return False
        padded = False
        if valid_token_mask is not None:
            if (tuple(valid_token_mask.shape) != tuple(x.shape[:2]) or valid_token_mask.device != x.device
                    or valid_token_mask.dtype not in (torch.bool, torch.uint8)):
                return False
            padded = not self._all_tokens_valid(valid_token_mask, x.shape[1])
            if padded and not valid_token_mask.is_contiguous():
                return False
        plan = self.execution_plan(x.shape[0], x.shape[1], padded=padded)
        chunk = self._large_batch_chunk_size or plan.batch_chunk_size  # the caller's (TTB:1740), else the plan's
        return plan.fused and not (chunk and x.shape[0] > chunk)

    def _all_tokens_valid(self, valid_token_mask: Optional[torch.Tensor], seq_len: int) -> bool:
        """Mask inspection cached by identity + version + length (TTB:464-522)."""
        if valid_token_mask is None:
            return True
        version = _tensor_version(valid_token_mask)
        cached = self.__dict__.get("_mask_cache")
        if version is not None and cached is not None and cached[0] is valid_token_mask and cached[1] == version and cached[2] == seq_len:
            return cached[3]
        result = bool(valid_token_mask.all().item())
        if version is not None:
            self.__dict__["_mask_cache"] = (valid_token_mask, version, seq_len, result)
        return result

    # ----------------------------------------------------------------- forward
    def forward(self, x: torch.Tensor, valid_token_mask: Optional[torch.Tensor] = None) -> torch.Tensor:
        return self._forward_impl(x, valid_token_mask, None)

    def _forward_into(self, x: torch.Tensor, out: torch.Tensor,
                      valid_token_mask: Optional[torch.Tensor] = None) -> torch.Tensor:
        """forward(x, valid_token_mask) written into `out` (contiguous float32, x's shape) and returned.

        BatchChunkedTransformer writes each chunk into its slice of the batch
        output this way, with no copy of a separately allocated result.
        """
        return self._forward_impl(x, valid_token_mask, out)

    def _forward_impl(self, x: torch.Tensor, valid_token_mask: Optional[torch.Tensor],
                      out: Optional[torch.Tensor]) -> torch.Tensor:
        if torch.is_grad_enabled():  # entering no_grad costs 1 us: only where it changes anything
            with torch.no_grad():
                return self._forward_impl(x, valid_token_mask, out)
        if x.device.type != "cuda":
            raise RuntimeError(
                "UserOptimizedTransformer runs only on the gfx950 HIP path; move the model and "
                "input to the GPU (there is deliberately no CPU fallback)"
            )
        if self._mixed_precision_dtype != torch.float16:
            raise NotImplementedError("the gfx950 path implements float16 compute only")
        if x.ndim != 3 or x.shape[-1] != self.config.d_model:
            raise ValueError(f"expected input [B, S, {self.config.d_model}], got {tuple(x.shape)}")
        if x.dtype != torch.float32:
            raise ValueError("the gfx950 path expects a float32 residual stream input")
        if self.training:
            raise RuntimeError("UserOptimizedTransformer is inference-only; call eval()")
        if out is not None and (tuple(out.shape) != tuple(x.shape) or out.dtype != torch.float32
                                or out.device != x.device or not out.is_contiguous()):
            raise ValueError(f"out must be a contiguous float32 tensor of shape {tuple(x.shape)} on {x.device}")
        token_valid = None
        if valid_token_mask is not None:
            if tuple(valid_token_mask.shape) != tuple(x.shape[:2]):
                raise ValueError(
                    f"valid_token_mask must be [B, S] = {tuple(x.shape[:2])}, got {tuple(valid_token_mask.shape)}")
            if valid_token_mask.device != x.device:
                raise ValueError("valid_token_mask must be on the input's device")
            if valid_token_mask.dtype not in (torch.bool, torch.uint8):
                raise ValueError("valid_token_mask must be bool or uint8")
            if x.numel() and not self._all_tokens_valid(valid_token_mask, x.shape[1]):
                # Every kernel tests the mask's bytes against zero, so a bool mask is read
                # as it is: converting it first took two launches, 11 us of a 51 us forward.
                token_valid = valid_token_mask.contiguous().view(torch.uint8)
        if x.numel() == 0:  # no sequence or no token: an empty result, nothing launched, no cache change
            return torch.empty_like(x) if out is None else out
        x = x.contiguous()
        if self._kv_cache_enabled:
            if token_valid is not None:
                raise ValueError("KV-cached decoding does not support padding")
            result = self._forward_hip_cached(x)
            return result if out is None else out.copy_(result)
        plan = self.execution_plan(x.shape[0], x.shape[1], padded=token_valid is not None)
        chunk = self._large_batch_chunk_size or plan.batch_chunk_size
        if chunk and x.shape[0] > chunk:
            output = torch.empty_like(x) if out is None else out
            for start in range(0, x.shape[0], chunk):
                end = min(start + chunk, x.shape[0])
                self._forward_hip(x[start:end], out=output[start:end],
                                  token_valid=None if token_valid is None else token_valid[start:end])
            return output
        return self._forward_hip(x, out=out, token_valid=token_valid, plan=plan)

    def _forward_hip(self, x: torch.Tensor, out: Optional[torch.Tensor] = None,
                     token_valid: Optional[torch.Tensor] = None,
                     plan: Optional[ShapeExecutionPlan] = None) -> torch.Tensor:
        """The fused kernel sequence of TTB:1092-1148 for one batch.

        token_valid: None (every token valid) or a contiguous [B, S] uint8 mask
        with at least one zero.  plan: execution_plan(B, S, padded=token_valid
        is not None) when the caller already has it.
        """
        cfg = self.config
        if plan is None:
            plan = self.execution_plan(x.shape[0], x.shape[1], padded=token_valid is not None)
        if not plan.runnable:
            raise ValueError(f"no gfx950 kernel sequence for this input: {plan.forward_strategy}")
        if plan.fused:
            wpack, ppack, affine_mask = self._fused_stack_parameters()
            return kernels.fused_forward_d128(x, wpack, ppack, cfg.num_heads, cfg.ffn_dim, len(self.layers), out=out,
                                              affine_mask=affine_mask, token_valid=token_valid, causal=cfg.causal,
                                              split=plan.fused_variant == _capi.XB_FUSED_SPLIT,
                                              strict=self._strict_handoff_checks)

        return self._per_op_forward(x, plan, out=out, token_valid=token_valid)

    def captured_overlap(self, batch: int, seq_len: int, padded: bool = False) -> Optional[str]:
        """What a captured forward of [batch, seq_len] runs beyond its plan: None, the plan's launches on one stream.

        Two half-batches on two streams are slower at every size tried (us per replay, two
        streams / one: 64 x 128 tokens of width 1024, 4 layers 684 / 663; 16 x 512, width 768,
        2 layers 415 / 376; 4 x 128, width 256, 4 layers 285 / 112): the GEMM tiles already put
        two blocks on a CU, and a graph with two branches costs more per launch.
        """
        return None

    def _forward_hip_cached(self, x: torch.Tensor) -> torch.Tensor:
        """One KV-cached step: append this chunk's keys/values per layer, attend over the cache.

        Caches are [B, H, config.seq_len, hd] FP16 per layer, allocated on the
        first step (TTB:426-462).  The prompt (position 0) attends within its
        own projection; later chunks read the cache, decode-sized ones (<= 16
        tokens) through the split-key kernel.
        """
        cfg = self.config
        batch, chunk, _ = x.shape
        start = self._kv_cache_length
        capacity = cfg.seq_len
        if start + chunk > capacity:
            raise ValueError(f"KV cache capacity exceeded ({start + chunk} > {capacity})")
        expected = (batch, cfg.num_heads, capacity, cfg.head_dim)
        for index in range(len(self.layers)):
            cached = self._kv_cache.get(index)
            if cached is None:
                self._kv_cache[index] = tuple(
                    torch.empty(expected, device=x.device, dtype=torch.float16) for _ in range(2))
            elif tuple(cached[0].shape) != expected or cached[0].device != x.device:
                raise RuntimeError(
                    "KV cache does not match this input; reset it before changing batch size, device, or dtype")
        plan = self.execution_plan(batch, chunk, per_op=True)
        if not plan.runnable:
            raise ValueError(f"no gfx950 kernel sequence for this input: {plan.forward_strategy}")
        output = self._per_op_forward(x, plan, cache_start=start)
        self._kv_cache_length = start + chunk
        return output

    def _per_op_forward(self, x: torch.Tensor, plan: ShapeExecutionPlan, out: Optional[torch.Tensor] = None,
                        token_valid: Optional[torch.Tensor] = None, cache_start: Optional[int] = None) -> torch.Tensor:
        """LN -> per layer (QKV GEMM, attention, out GEMM, residual LN, FFN) -> final LN, issued natively.

        cache_start: None, or the position in the KV cache of x's first token.
        While a LaunchRecorder is active the same sequence goes through the
        wrappers one by one, so that each launch is bracketed by its events
        (a few rows' LayerNorms and cache appends are then launches of their
        own, with the same bits).
        """
        if plan.row_block and self.config.d_model == 32 and x.data_ptr() % 16:
            x = x.clone()  # this width's LayerNorm takes any alignment, the row blocks 16 bytes
        native = None if kernels.recording() else self._native_stack(plan.row_block)
        if native is None or native[3] != x.get_device():
            return self._per_op_forward_stepwise(x, plan, out, token_valid, cache_start)
        if out is None:
            out = torch.empty_like(x)
        variants = (plan.qkv_variant, plan.out_variant, plan.ffn_in_variant, plan.ffn_out_variant,
                    plan.attention_variant)
        if cache_start is None:
            return kernels.stack_forward(x, native[0], variants, out, token_valid=token_valid)
        pointers = [t.data_ptr() for index in range(len(self.layers)) for t in self._kv_cache[index]]
        return kernels.stack_forward(x, native[0], variants, out, caches=(ctypes.c_void_p * len(pointers))(*pointers),
                                     cache_start=cache_start, cache_capacity=self.config.seq_len)

    def _attend_stepwise(self, index: int, qkv: torch.Tensor, plan: ShapeExecutionPlan,
                         token_valid: Optional[torch.Tensor], cache_start: Optional[int]) -> torch.Tensor:
        heads, scale = self.config.num_heads, self.layers[index].attention.scale
        if cache_start is not None:
            k_cache, v_cache = self._kv_cache[index]
            kernels.kv_cache_append(qkv, k_cache, v_cache, heads, cache_start)
            if cache_start:
                return kernels.attention_kv_cache(qkv, k_cache, v_cache, heads, cache_start, scale=scale)
        return kernels.attention(qkv, heads, key_valid=token_valid, causal=self.config.causal, scale=scale,
                                 variant=plan.attention_variant)

    def _per_op_forward_stepwise(self, x: torch.Tensor, plan: ShapeExecutionPlan, out: Optional[torch.Tensor],
                                 token_valid: Optional[torch.Tensor], cache_start: Optional[int]) -> torch.Tensor:
        """_per_op_forward, one wrapper call per launch."""
        native = self._native_stack(True) if plan.row_block else None
        if native is not None and native[3] == x.get_device():
            return self._row_block_forward_stepwise(x, native[0], plan, out, token_valid, cache_start)
        cfg = self.config
        batch, seq_len, d_model = x.shape
        dev = x.device
        f16 = torch.float16
        num_layers = len(self.layers)

        # The long-sequence attention reading V transposed by the QKV GEMM
        # (one buffer for all layers).
        transposed_v = plan.attention_variant == _capi.XB_ATTN_PINGPONG_VT
        vt = None
        if transposed_v:
            vt = torch.empty((batch, cfg.num_heads, cfg.head_dim, kernels.vt_row_stride(seq_len)), device=dev,
                             dtype=torch.float16)
        first = self.layers[0].norm1
        norm = kernels.layer_norm(x, first.weight, first.bias, first.eps, f16, apply_affine=self._layer_norm_uses_affine(first))
        residual_in = x
        residual = torch.empty((batch, seq_len, d_model), device=dev, dtype=torch.float32)
        if out is None:
            out = torch.empty_like(x)
        for index, layer in enumerate(self.layers):
            w = self._layer_weights(index)
            if transposed_v:
                qkv, _ = kernels.linear_qkv_vt(norm, w.qkv_w, w.qkv_b, cfg.num_heads, vt=vt, variant=plan.qkv_variant)
                context = kernels.attention_vt(qkv, vt, cfg.num_heads, scale=layer.attention.scale)
            else:
                qkv = kernels.linear(norm, w.qkv_w, w.qkv_b, variant=plan.qkv_variant)
                context = self._attend_stepwise(index, qkv, plan, token_valid, cache_start)
            update = kernels.linear(context, w.out_w, w.out_b, variant=plan.out_variant)
            residual_in, norm2 = kernels.fused_residual_layer_norm(
                residual_in, update, layer.norm2.weight, layer.norm2.bias, layer.norm2.eps, f16,
                apply_affine=self._layer_norm_uses_affine(layer.norm2), residual_out=residual,
            )
            planned = w.ffn_in_w.shape[0] == cfg.ffn_dim  # the plan's tiles are for the config's width
            hidden = kernels.linear(norm2, w.ffn_in_w, w.ffn_in_b, gelu=True,
                                    variant=plan.ffn_in_variant if planned else _capi.XB_VARIANT_AUTO)
            update = kernels.linear(hidden, w.ffn_out_w, w.ffn_out_b,
                                    variant=plan.ffn_out_variant if planned else _capi.XB_VARIANT_AUTO)
            last = index == num_layers - 1
            following = self.final_norm if last else self.layers[index + 1].norm1
            residual_in, norm = kernels.fused_residual_layer_norm(
                residual_in, update, following.weight, following.bias, following.eps,
                torch.float32 if last else f16, store_residual=not last,
                apply_affine=self._layer_norm_uses_affine(following),
                residual_out=residual, norm_out=out if last else None,
                row_valid=token_valid if last else None,
                mask_mode=_capi.XB_MASK_OUTPUT if last and token_valid is not None else 0,
            )
        return norm

    def _row_block_forward_stepwise(self, x: torch.Tensor, stack: _capi.XbStack, plan: ShapeExecutionPlan,
                                    out: Optional[torch.Tensor], token_valid: Optional[torch.Tensor],
                                    cache_start: Optional[int]) -> torch.Tensor:
        if out is None:
            out = torch.empty_like(x)
        qkv = torch.empty((*x.shape[:2], 3 * x.shape[2]), device=x.device, dtype=torch.float16)
        kernels.row_block(stack, -1, x, qkv=qkv)
        residual = x
        for index in range(len(self.layers)):
            context = self._attend_stepwise(index, qkv, plan, token_valid, cache_start)
            last = index == len(self.layers) - 1
            updated = None if last else torch.empty_like(x)
            kernels.row_block(stack, index, residual, ctx=context, residual_out=updated, qkv=None if last else qkv,
                              out=out if last else None, row_valid=token_valid if last else None)
            residual = updated
        return out


def forward_flops(config: TransformerConfig, batch: Optional[int] = None, seq_len: Optional[int] = None) -> float:
    """GEMM + causal-attention FLOPs of one forward (2*B*S*L*(4D^2+2DF) + 2*B*L*D*S*(S+1))."""
    b = config.batch_size if batch is None else batch
    s = config.seq_len if seq_len is None else seq_len
    d, f, layers = config.d_model, config.ffn_dim, config.num_layers
    return 2.0 * b * s * layers * (4 * d * d + 2 * d * f) + 2.0 * b * layers * d * s * (s + 1)


def forward_bytes(config: TransformerConfig, batch: Optional[int] = None, seq_len: Optional[int] = None) -> float:
    """HBM bytes of the unfused kernel pipeline: B*S*(4D + L*(48D + 4F)) + 2*L*(4D^2 + 2DF)."""
    b = config.batch_size if batch is None else batch
    s = config.seq_len if seq_len is None else seq_len
    d, f, layers = config.d_model, config.ffn_dim, config.num_layers
    return b * s * (4 * d + layers * (48 * d + 4 * f)) + 2.0 * layers * (4 * d * d + 2 * d * f)


__all__ = [
    "SelfAttentionParameters",
    "TransformerBlockParameters",
    "UserOptimizedTransformer",
    "forward_flops",
    "forward_bytes",
]
