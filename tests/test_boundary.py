"""CPU tests of the drop-in boundary: config type, state_dict compatibility,
the C-ABI library's exports and argument checks, and the no-fallback rule."""

from __future__ import annotations

import ctypes
import json
import re
from pathlib import Path

import pytest
import torch

from oracle.baseline import BaselineTransformer, copy_model_weights

REPO = Path(__file__).resolve().parents[1]


def test_config_validation_messages(pkg):
    TC = pkg.TransformerConfig
    TC(2, 4, 8, 2, 8, 1, True).validate()
    with pytest.raises(ValueError, match="batch_size must be positive"):
        TC(0, 4, 8, 2, 8, 1, True).validate()
    with pytest.raises(ValueError, match=r"d_model \(10\) must be divisible by num_heads \(4\)"):
        TC(1, 4, 10, 4, 8, 1, True).validate()
    with pytest.raises(ValueError, match="num_layers must be positive"):
        TC(1, 4, 8, 2, 8, 0, True).validate()
    assert hash(TC(1, 2, 8, 2, 8, 1, True)) == hash(TC(1, 2, 8, 2, 8, 1, True))


def test_benchmark_configs_match_baseline_json(pkg):
    """BASELINE.json's five configs are official shapes 1, 6, 8, 11, 14."""
    configs = json.loads((REPO / "BASELINE.json").read_text())["configs"]
    assert len(configs) == 5
    expected = [(64, 128, 128, 4, 128, 4), (10000, 128, 128, 4, 128, 4), (64, 128, 1024, 4, 1024, 4),
                (64, 128, 128, 16, 128, 4), (32, 100000, 1024, 16, 1024, 2)]
    for shape_id, geom in zip(pkg.BENCHMARK_CONFIG_SHAPE_IDS, expected):
        c = pkg.OFFICIAL_BENCHMARK_SHAPES[shape_id]
        assert (c.batch_size, c.seq_len, c.d_model, c.num_heads, c.ffn_dim, c.num_layers) == geom
        assert c.causal
    assert "B=10000" in configs[1] and "head_dim 8" in configs[3] and "S=100000" in configs[4]


def test_shape_plan(pkg, capi):
    """The plan is the library's selection (no GPU needed) and names what runs."""
    shapes = pkg.OFFICIAL_BENCHMARK_SHAPES
    plan = pkg.resolve_shape_execution_plan(shapes[6])
    assert plan.official_shape_id == 6
    assert plan.describe().startswith("official-6: ffn=")
    assert plan.fused and plan.fused_variant == capi.XB_FUSED_PAIRS and plan.batch_chunk_size == 0
    assert "fused_stack_1wg_8wave_pairs" in plan.describe()
    # small causal batches (up to 128 sequences) split each sequence over two workgroups
    for shape_id in (1, 5, 11):
        assert pkg.resolve_shape_execution_plan(shapes[shape_id]).fused_variant == capi.XB_FUSED_SPLIT
    # D=1024: per-op kernels; the QKV GEMM's tile is the cost model's (256 x 192 for N = 3072)
    cfg3 = pkg.resolve_shape_execution_plan(shapes[8])
    assert not cfg3.fused and cfg3.qkv_variant == 1 and "mfma_gemm_dma_256x192" in cfg3.projection_strategy
    assert "2x128x192" in cfg3.projection_strategy                                # the blocks that it launches
    assert cfg3.attention_strategy == "flash_8wave_128q"
    cfg5 = pkg.resolve_shape_execution_plan(shapes[14])
    assert cfg5.attention_strategy == "flash_pingpong_vt_8wave_512q" and cfg5.batch_chunk_size == 0
    assert cfg5.attention_variant == capi.XB_ATTN_PINGPONG_VT and cfg5.qkv_variant == capi.XB_LINEAR_DMA_256x256
    # V transposed by the QKV GEMM needs 32 | S and is not used for KV-cached steps
    odd = pkg.TransformerConfig(2, 100001, 1024, 16, 1024, 2, True)
    assert pkg.resolve_shape_execution_plan(odd).attention_strategy == "flash_pingpong_8wave_512q"
    assert pkg.resolve_shape_execution_plan(shapes[14], transposed_v_allowed=False).attention_variant == \
        capi.XB_ATTN_PINGPONG
    # a padded mask takes the key-masked forms: no ping-pong kernel
    assert pkg.resolve_shape_execution_plan(shapes[14], masked=True).attention_strategy == "flash_4wave_256q"
    # the whole-stack kernel off (toggle or LayerNorm contract): per-op
    assert not pkg.resolve_shape_execution_plan(shapes[6], fused_allowed=False).fused
    # a batch beyond the HBM budget runs in slices
    big = pkg.TransformerConfig(400, 100000, 1024, 16, 1024, 2, True)
    chunked = pkg.resolve_shape_execution_plan(big)
    assert 0 < chunked.batch_chunk_size < 400 and "batch_chunk=" in chunked.describe()
    # up to 8 rows of some widths: LayerNorms inside the products
    few = pkg.TransformerConfig(4, 2, 1024, 16, 1024, 2, True)
    assert "LayerNorm inside the QKV GEMM" in pkg.resolve_shape_execution_plan(few).describe()
    for more in (pkg.TransformerConfig(9, 1, 1024, 16, 1024, 2, True), pkg.TransformerConfig(4, 2, 256, 4, 256, 2, True)):
        assert "per_op (LayerNorm, QKV GEMM" in pkg.resolve_shape_execution_plan(more).describe()
    general = pkg.resolve_shape_execution_plan(pkg.TransformerConfig(3, 5, 8, 2, 8, 1, True))
    assert general.official_shape_id is None and general.describe().startswith("general:")


def test_variant_selection_abi(capi):
    """xb_select_* and the *_v entry points' variant checks need no GPU."""
    lib = capi.lib()
    assert lib.xb_select_linear(8192, 3072, 1024, 0) == 1          # 256 x 192
    assert lib.xb_select_linear(8192, 384, 128, 0) in (4, 5)       # K = 128: the nt kernel
    assert lib.xb_select_linear(-1, 8, 8, 0) == -2
    assert lib.xb_select_attention(64, 128, 4, 256, 0) == 3          # cfg3: one 8-wave block per (batch, head)
    assert lib.xb_select_attention(8, 128, 4, 256, 0) == 0           # too few blocks for that
    assert lib.xb_select_attention(32, 100000, 16, 64, 0) == 4
    assert lib.xb_select_attention(32, 100000, 16, 64, 1) == 2
    # head_dim 64 without a mask: the ping-pong kernel from 16384 queries on, from 12288 with 32 heads
    for batch, s, variant in ((2, 4128, 1), (2, 12287, 1), (4, 12287, 2), (2, 12288, 4), (1, 12288, 1), (1, 16384, 4)):
        assert lib.xb_select_attention(batch, s, 16, 64, 0) == variant, (batch, s)
    assert lib.xb_select_attention(1, 8, 2, 24, 0) == -4
    assert lib.xb_select_fused_d128(64, 128, 4, 128, 1, 0) == 1
    assert lib.xb_select_fused_d128(10000, 128, 4, 128, 1, 0) == 0
    assert lib.xb_select_fused_d128(8, 128, 1, 128, 1, 1) == -4    # head_dim 128: causal, unmasked only
    assert lib.xb_select_fused_d128(8, 129, 4, 128, 1, 0) == -4
    # a variant not built for the shape is refused before any launch
    assert lib.xb_linear_v(16, 16, None, 16, 8192, 384, 128, 0, 0, None) == -10      # DMA tile needs K >= 256
    assert lib.xb_linear_v(16, 16, None, 16, 8192, 1024, 1024, 0, 1, None) == -10    # 256 x 192 needs N % 192
    assert lib.xb_attention_v(16, 16, None, 2, 64, 2, 32, 0.1, 1, 4, None) == -10     # ping-pong: head_dim 64 only
    assert lib.xb_attention_v(16, 16, 16, 2, 64, 2, 64, 0.1, 1, 4, None) == -10       # nor with a key mask
    names = {lib.xb_variant_name(op, v) for op, n in ((0, 8), (1, 6), (2, 3)) for v in range(n)}
    assert None not in names and len(names) == 17
    assert lib.xb_variant_name(0, 99) is None


@pytest.mark.parametrize("geom", [(2, 8, 32, 4, 48, 2), (1, 4, 128, 16, 128, 1)])
def test_state_dict_is_the_baselines(pkg, geom):
    cfg = pkg.TransformerConfig(*geom, True)
    torch.manual_seed(1234)
    baseline = BaselineTransformer(cfg)
    torch.manual_seed(1234)
    optimized = pkg.UserOptimizedTransformer(cfg)
    assert list(baseline.state_dict().keys()) == list(optimized.state_dict().keys())
    # Same construction order => the same seeded nn.Linear initialisation.
    for (k, a), (_, b) in zip(baseline.state_dict().items(), optimized.state_dict().items()):
        assert torch.equal(a, b), k
    other = pkg.UserOptimizedTransformer(cfg)
    copy_model_weights(baseline, other)  # strict load_state_dict (TTB:1151-1161)
    for (k, a), (_, b) in zip(baseline.state_dict().items(), other.state_dict().items()):
        assert torch.equal(a, b), k


def test_forward_has_no_cpu_fallback(pkg):
    cfg = pkg.TransformerConfig(1, 4, 32, 4, 32, 1, True)
    model = pkg.UserOptimizedTransformer(cfg).eval()
    with pytest.raises(RuntimeError, match="no CPU fallback"):
        model(torch.randn(1, 4, 32))


def test_toggles(pkg):
    model = pkg.UserOptimizedTransformer(pkg.TransformerConfig(1, 4, 32, 4, 32, 1, True))
    with pytest.raises(ValueError):
        model.enable_mixed_precision(torch.float32)
    model.enable_mixed_precision(torch.float16)
    with pytest.raises(RuntimeError, match="eval"):
        model.enable_kv_cache(True)           # still in training mode (TTB:412-413)
    model.eval().enable_kv_cache(True)
    assert model.kv_cache_length == 0
    model.enable_kv_cache(False)
    assert model.kv_cache_length == 0
    with pytest.raises(ValueError, match="causal"):
        pkg.UserOptimizedTransformer(pkg.TransformerConfig(1, 4, 32, 4, 32, 1, False)).eval().enable_kv_cache(True)
    assert model.shape_execution_plan.official_shape_id is None
    # The reference's main() toggles (TTB:1765-1770) are accepted.
    model.enable_triton_fused_norm(False)
    model.enable_triton_fused_ffn(False)
    model.enable_attention_fp16_accumulation(False)
    with pytest.raises(ValueError, match="causal"):
        model.enable_attention_fp16_accumulation(True)
    pkg.UserOptimizedTransformer(pkg.TransformerConfig(1, 4, 32, 4, 32, 1, False)).enable_attention_fp16_accumulation(True)


def test_tree_cache_follows_registrations(pkg):
    """The cached parameter / LayerNorm walk is redone after any parameter or module assignment."""
    model = pkg.UserOptimizedTransformer(pkg.TransformerConfig(2, 8, 128, 4, 128, 2, True)).eval()
    x = torch.empty(2, 8, 128)
    params, norms = model._tree()
    assert list(params) == list(model.parameters()) and len(norms) == 2 * 2 + 1
    assert model._tree()[0] is params                      # no registration: the same walk
    assert model._fused_stack_eligible() and not model._single_launch_forward(x, None)  # CPU input
    fresh = torch.nn.Parameter(torch.zeros(128, 128))
    model.layers[1].ffn_in.weight = fresh
    assert any(p is fresh for p in model._tree()[0])
    model.final_norm = torch.nn.LayerNorm(128, eps=1e-6)
    assert model._tree()[1][-1] is model.final_norm
    assert not model._fused_stack_eligible()               # eps outside the kernel's contract
    assert not model.execution_plan(2, 8).fused


@pytest.mark.parametrize("change", ["del", "pop", "insert", "swap"])
def test_native_descriptor_follows_the_layers(pkg, change):
    """The native sequence runs the layers that the model has now: modules that leave or
    enter without a registration hook are in the next descriptor, as the live loop had them."""
    model = pkg.UserOptimizedTransformer(pkg.TransformerConfig(2, 300, 256, 4, 256, 3, True)).eval()
    assert model._native_stack(False)[0].layers == 3
    layers = model.layers
    if change == "del":
        del layers[2]
    elif change == "pop":
        layers.pop(0)
    elif change == "insert":
        layers.insert(1, layers[2])
    else:
        layers[1]._modules["ffn_in"] = torch.nn.Linear(256, 256)
    stack, blocks, _ = model._native_stack(False)[:3]
    assert stack.layers == len(blocks) == len(layers)
    for block, layer in zip(blocks, layers):
        assert block.norm1_g == layer.norm1.weight.data_ptr()
    assert blocks[1].ffn_in_w == model._layer_weights(1).ffn_in_w.data_ptr()
    assert all(any(p is q for q in model._tree()[0]) for p in layers[1].parameters())


def test_model_copies_and_saves_after_a_forward(pkg):
    """copy.deepcopy and torch.save work once the native descriptor exists; the copy keeps
    the settings and builds a descriptor of its own parameters."""
    import copy
    import io

    model = pkg.UserOptimizedTransformer(pkg.TransformerConfig(2, 300, 256, 4, 256, 2, True)).eval()
    model.enable_fused_stack(False)
    model._native_stack(False)
    file = io.BytesIO()
    torch.save(model, file)
    file.seek(0)
    for twin in (copy.deepcopy(model), torch.load(file, weights_only=False)):
        assert twin._fused_stack_enabled is False and not twin.training
        for p, q in zip(model.parameters(), twin.parameters()):
            assert torch.equal(p, q) and p.data_ptr() != q.data_ptr()
        _, blocks, weights = twin._native_stack(False)[:3]
        assert blocks[1].norm1_g == twin.layers[1].norm1.weight.data_ptr()
        assert torch.equal(weights[1].ffn_in_w, model.layers[1].ffn_in.weight.half())


@pytest.mark.parametrize("misfit", ["narrow_ffn", "wide_ffn", "norm", "final_norm", "half_norm", "projection", "bias"])
def test_native_descriptor_only_for_parameters_of_the_configs_sizes(pkg, misfit):
    """The native kernels take every size from the config: a parameter of another size, or a
    LayerNorm that isn't float32, gives no descriptor (the wrappers then run it or raise)."""
    model = pkg.UserOptimizedTransformer(pkg.TransformerConfig(2, 300, 256, 4, 512, 2, True)).eval()
    layer = model.layers[1]
    assert model._native_stack(False)[0].ffn_dim == 512
    if misfit.endswith("ffn"):
        width = 256 if misfit == "narrow_ffn" else 1024
        layer.ffn_in, layer.ffn_out = torch.nn.Linear(256, width), torch.nn.Linear(width, 256)
    elif misfit == "norm":
        layer.norm2 = torch.nn.LayerNorm(64)
    elif misfit == "final_norm":
        model.final_norm = torch.nn.LayerNorm(512)
    elif misfit == "half_norm":
        layer.norm1.half()
    elif misfit == "projection":
        layer.attention.k_proj = torch.nn.Linear(256, 64)
    else:
        layer.ffn_in.bias = None
    assert model._native_stack(False) is None and model._native_stack(True) is None
    assert model._native_stack(False) is None


def test_packed_weights_outlive_a_change_of_settings(pkg, monkeypatch):
    """Row-block weights belong to the parameters, not to the descriptor: a LayerNorm eps, the
    attention scale and the path toggle leave them where a captured graph reads them."""
    import importlib

    kernels = importlib.import_module(pkg.__name__ + ".kernels")
    monkeypatch.setattr(kernels, "pack_linear_fragments", lambda w, out: out.copy_(w.detach().flatten()))
    model = pkg.UserOptimizedTransformer(pkg.TransformerConfig(2, 300, 64, 4, 64, 2, True)).eval()
    packed = [w.packed for w in model._native_stack(True)[2]]
    model.layers[0].norm2.eps = 0.25
    model._native_stack(True)
    model.layers[1].attention.scale = 0.5
    model._native_stack(True)
    model._native_stack(False)                        # the per-op form between two row-block ones
    held = [entry[1] for entry in model._weight_cache.values()]
    assert all(any(getattr(w, "packed", None) is p for w in held) for p in packed)
    again = model._native_stack(True)
    assert all(w.packed is p for w, p in zip(again[2], packed))
    assert again[1][0].norm2_eps == 0.25 and again[1][1].scale == 0.5
    with torch.no_grad():
        model.layers[0].ffn_in.weight.add_(1.0)
    changed = [w.packed for w in model._native_stack(True)[2]]
    assert changed[0] is not packed[0] and changed[1] is packed[1]


def test_caches_of_an_older_file_are_dropped(pkg):
    """A model pickled with its derived caches inside loads without them: their form is not this code's."""
    model = pkg.UserOptimizedTransformer(pkg.TransformerConfig(2, 300, 256, 4, 256, 1, True)).eval()
    walk = (0, tuple(model.parameters()), tuple(m for m in model.modules() if isinstance(m, torch.nn.LayerNorm)))
    loaded = pkg.UserOptimizedTransformer.__new__(pkg.UserOptimizedTransformer)
    loaded.__setstate__({**model.__getstate__(), "_tree_cache": walk, "_weight_cache": {0: ((), None)}})
    assert "_tree_cache" not in loaded.__dict__ and "_weight_cache" not in loaded.__dict__
    assert loaded._native_stack(False)[0].layers == 1


def test_stack_forward_wants_two_caches_per_layer(pkg, monkeypatch):
    """The native sequence reads two cache pointers per layer: fewer are refused before the call."""
    import importlib

    kernels = importlib.import_module(pkg.__name__ + ".kernels")
    monkeypatch.setattr(kernels, "_require_device", lambda tensor, what: None)
    model = pkg.UserOptimizedTransformer(pkg.TransformerConfig(2, 8, 256, 4, 256, 2, True)).eval()
    x = torch.zeros(2, 8, 256)
    with pytest.raises(ValueError, match="2 layers need 4 cache pointers, got 2"):
        kernels.stack_forward(x, model._native_stack(False)[0], (-1,) * 5, torch.empty_like(x),
                              caches=(ctypes.c_void_p * 2)(16, 16), cache_capacity=8)


def test_native_descriptor_follows_functional_call(pkg):
    """Parameters swapped in for one call (torch.func.functional_call) are the ones it reads,
    and the model's own ones are back afterwards."""
    model = pkg.UserOptimizedTransformer(pkg.TransformerConfig(2, 300, 256, 4, 256, 1, True)).eval()
    own = model._native_stack(False)[1][0]
    seen = []
    model.forward = lambda: seen.append(model._native_stack(False))
    swapped = {name: p.detach() + 1.0 for name, p in model.named_parameters()}
    torch.func.functional_call(model, swapped, ())
    block, weights = seen[0][1][0], seen[0][2][0]
    assert block.norm1_g == swapped["layers.0.norm1.weight"].data_ptr() != own.norm1_g
    assert torch.equal(weights.out_w, swapped["layers.0.attention.out_proj.weight"].half())
    assert model._native_stack(False)[1][0].norm1_g == own.norm1_g == model.layers[0].norm1.weight.data_ptr()


def test_whole_stack_parameters_follow_functional_call(pkg, monkeypatch):
    """The whole-stack form packs the parameters of the call as well."""
    import importlib

    kernels = importlib.import_module(pkg.__name__ + ".kernels")
    monkeypatch.setattr(kernels, "pack_linear_fragments", lambda w, scale: (w.detach() * scale).half().flatten())
    model = pkg.UserOptimizedTransformer(pkg.TransformerConfig(2, 64, 128, 4, 128, 1, True)).eval()
    own = model._fused_stack_parameters()
    assert model._fused_stack_parameters()[0] is own[0]
    seen = []
    model.forward = lambda: seen.append(model._fused_stack_parameters())
    swapped = {name: p.detach() + 1.0 for name, p in model.named_parameters()}
    torch.func.functional_call(model, swapped, ())
    assert not torch.equal(seen[0][0], own[0]) and not torch.equal(seen[0][1], own[1])
    assert torch.equal(seen[0][1][-256:-128], swapped["final_norm.weight"])
    again = model._fused_stack_parameters()
    assert torch.equal(again[0], own[0]) and torch.equal(again[1], own[1])


@pytest.mark.parametrize("form", ["native", "whole_stack"])
def test_cached_addresses_stay_taken(pkg, monkeypatch, form):
    """What was derived from tensors swapped in for one call is keyed by their addresses, so
    they stay alive until it is replaced: the next call's cannot lie where they lay."""
    import importlib
    import weakref

    kernels = importlib.import_module(pkg.__name__ + ".kernels")
    monkeypatch.setattr(kernels, "pack_linear_fragments", lambda w, scale=1.0: (w.detach() * scale).half().flatten())
    d = 128 if form == "whole_stack" else 256
    model = pkg.UserOptimizedTransformer(pkg.TransformerConfig(2, 64, d, 4, d, 1, True)).eval()
    derive = model._fused_stack_parameters if form == "whole_stack" else lambda: model._native_stack(False)
    model.forward = derive
    swapped = {name: p.detach() + 1.0 for name, p in model.named_parameters()}
    refs = [weakref.ref(t) for t in swapped.values()]
    torch.func.functional_call(model, swapped, ())
    del swapped
    assert all(ref() is not None for ref in refs)
    derive()
    assert all(ref() is None for ref in refs)


def test_native_descriptor_only_for_its_own_norms(pkg):
    """A parametrized LayerNorm weight is another tensor on each access: no descriptor points at one."""
    model = pkg.UserOptimizedTransformer(pkg.TransformerConfig(2, 64, 256, 4, 256, 1, True)).eval()
    torch.nn.utils.parametrize.register_parametrization(model.layers[0].norm2, "weight", torch.nn.Identity())
    assert model._native_stack(False) is None
    weight = model.layers[0].attention.out_proj
    torch.nn.utils.parametrize.remove_parametrizations(model.layers[0].norm2, "weight")
    torch.nn.utils.parametrize.register_parametrization(weight, "weight", torch.nn.Identity())
    stack, _, weights = model._native_stack(False)[:3]     # a projection's is copied
    assert torch.equal(weights[0].out_w, weight.weight.half())


def test_native_descriptor_follows_the_config(pkg):
    """The descriptor's causal flag and the plans are the present config's."""
    import dataclasses

    model = pkg.UserOptimizedTransformer(pkg.TransformerConfig(2, 300, 256, 4, 256, 1, True)).eval()
    assert model._native_stack(False)[0].causal == 1
    assert "pingpong_vt" in model.execution_plan(8, 12288).attention_strategy
    model.config = dataclasses.replace(model.config, causal=False)
    assert model._native_stack(False)[0].causal == 0
    assert model.execution_plan(8, 12288).attention_strategy == "flash_pingpong_8wave_512q"   # V^T is for causal only


def test_fused_eligibility_checks_every_layer_norm_on_each_call(pkg):
    """The whole-stack kernel needs eps 1e-5, a weight and a bias on every LayerNorm, re-read per call."""
    model = pkg.UserOptimizedTransformer(pkg.TransformerConfig(2, 8, 128, 4, 128, 2, True)).eval()
    assert model._fused_stack_eligible() and model.execution_plan(2, 8).fused
    model.layers[0].norm2.eps = 1e-6                       # a plain attribute: no registration hook fires
    assert not model._fused_stack_eligible() and not model.execution_plan(2, 8).fused
    model.layers[0].norm2.eps = 1e-5
    assert model._fused_stack_eligible() and model.execution_plan(2, 8).fused
    for replacement in (torch.nn.LayerNorm(128, elementwise_affine=False), torch.nn.LayerNorm(128, bias=False)):
        model.layers[1].norm1 = replacement                # weight or bias registered as None
        assert not model._fused_stack_eligible()
    model.layers[1].norm1 = torch.nn.LayerNorm(128)
    assert model._fused_stack_eligible()
    model.enable_fused_stack(False)
    assert not model._fused_stack_eligible() and not model.execution_plan(2, 8).fused


def test_product_never_touches_the_oracle():
    for path in (REPO / "gpu-kernel-for-transformer_amd").rglob("*.py"):
        text = path.read_text()
        assert not re.search(r"^\s*(from|import)\s+oracle", text, re.M), path


# ----------------------------------------------------------------------------- C-ABI
def _declared_symbols():
    header = (REPO / "include" / "xblock.h").read_text()
    return sorted(set(re.findall(r"^\s*(?:int|int64_t|const char\*)\s+(xb_\w+)\s*\(", header, re.M)))


def test_library_exports_every_declared_symbol(capi):
    assert capi.XBLOCK_AVAILABLE, capi.XBLOCK_LOAD_ERROR
    declared = _declared_symbols()
    assert declared == sorted(capi.EXPORTED_SYMBOLS)
    handle = ctypes.CDLL(str(capi.LIBRARY_PATH))
    for name in declared:
        assert hasattr(handle, name), name
    assert capi.lib().xb_abi_version() == capi.XB_ABI_VERSION


SCRATCH_BYTES = 32 << 20   # XB_DECODE_SCRATCH_BYTES


def _check_noalloc_scratch_rule(lib):
    """The no-allocation decode's documented limit, from the library's own sizing.

    A decode chunk's partials (batch*heads*n_splits*16*(4*head_dim+8) bytes)
    fit the static scratch whenever one split per (batch, head) does, at any
    cache length; beyond that the call is refused (-9) before any launch.
    Only the refusals are called here: an accepted call would launch.
    """
    limits = {8: 52428, 16: 29127, 32: 15420, 64: 7943, 128: 4032, 256: 2032}
    for head_dim, limit in limits.items():
        assert limit == SCRATCH_BYTES // (16 * (4 * head_dim + 8))
        for bh in (1, 13, 16, 33, 48, 512, 2000, limit):
            for cached in (31, 4000, 100000):
                need = lib.xb_attention_kv_cache_workspace_bytes(bh, 1, 1, head_dim, cached)
                assert 0 < need <= SCRATCH_BYTES, (head_dim, bh, cached, need)
        for cached in (31, 100000):
            need = lib.xb_attention_kv_cache_workspace_bytes(limit + 1, 1, 1, head_dim, cached)
            assert need == (limit + 1) * 16 * (4 * head_dim + 8) > SCRATCH_BYTES
            assert lib.xb_attention_kv_cache_noalloc(16, 16, 16, 16, limit + 1, 1, 1, head_dim, cached,
                                                     cached + 1, 0.1, None) == -9
    # the long caches still split over many key ranges (a workspace call and
    # a no-allocation call share this geometry)
    assert lib.xb_attention_kv_cache_workspace_bytes(1, 1, 16, 256, 100000) > 100 * 16 * 16 * 1032


def test_argument_errors_need_no_gpu(capi):
    lib = capi.lib()
    assert lib.xb_linear(None, None, None, None, 4, 8, 8, 0, None) == -1
    assert lib.xb_linear(None, None, None, None, 0, 8, 8, 0, None) == 0   # empty: NULL allowed
    assert lib.xb_layernorm(None, None, None, None, 1, 0, 128, 1e-5, 0, None) == 0
    assert lib.xb_linear(16, 16, None, 16, 4, 7, 8, 0, None) == -4      # N % 8
    assert lib.xb_linear(16, 16, None, 16, 4, 8, 8, 9, None) == -6      # epilogue
    assert lib.xb_linear(18, 16, None, 16, 4, 8, 8, 0, None) == -5      # alignment
    assert lib.xb_linear(16, 16, None, 16, 0, 8, 8, 0, None) == 0       # empty: no launch
    assert lib.xb_layernorm(16, None, None, 16, 7, 4, 128, 1e-5, 0, None) == -3
    assert lib.xb_layernorm(16, None, None, 16, 1, -1, 128, 1e-5, 0, None) == -2
    assert lib.xb_layernorm(16, None, None, 16, 1, 4, 128, 1e-5, 1, None) == -1  # affine w/o gamma
    assert lib.xb_residual_layernorm(16, 16, 1, None, None, None, 16, 1, 0, 128, 1e-5, 0, None) == 0
    assert lib.xb_attention_causal(16, 16, 1, 8, 2, 24, 0.1, None) == -4  # head_dim 24
    assert lib.xb_attention_causal(16, 16, 0, 8, 2, 8, 0.1, None) == 0
    assert lib.xb_attention(16, 16, None, 1, 8, 2, 24, 0.1, 0, None) == -4   # head_dim 24
    assert lib.xb_attention(None, None, None, 1, 8, 2, 64, 0.1, 1, None) == -1
    assert lib.xb_attention(16, 16, None, 0, 8, 2, 64, 0.1, 0, None) == 0    # empty: no launch
    # KV cache: capacity, head_dim, workspace sizing without a GPU
    assert lib.xb_kv_cache_append(16, 16, 16, 1, 5, 2, 64, 10, 12, None) == -2   # 10 + 5 > 12
    assert lib.xb_kv_cache_append(16, 16, 16, 1, 5, 2, 24, 0, 12, None) == -4
    assert lib.xb_kv_cache_append(None, None, None, 1, 5, 2, 64, 0, 12, None) == -1
    assert lib.xb_attention_kv_cache_workspace_bytes(1, 17, 2, 64, 100) == 0     # long chunk: none needed
    assert lib.xb_attention_kv_cache_workspace_bytes(1, 1, 16, 64, 20000) == 7096320
    assert lib.xb_attention_kv_cache_workspace_bytes(1, 1, 2, 24, 100) == -4
    assert lib.xb_attention_kv_cache(16, 16, 16, 16, 1, 1, 2, 64, 100, 101, 0.1, None, 0, None) == -1
    assert lib.xb_attention_kv_cache(16, 16, 16, 16, 1, 1, 2, 64, 100, 101, 0.1, 16, 64, None) == -7
    # mask_mode outside UPDATE|SUM|OUTPUT, and a mask mode without row_valid
    assert lib.xb_residual_layernorm_masked(16, 16, 1, None, None, None, 16, 1, 4, 128, 1e-5, 0, 16, 8, None) == -6
    assert lib.xb_residual_layernorm_masked(16, 16, 1, None, None, None, 16, 1, 4, 128, 1e-5, 0, None, 2, None) == -1
    assert lib.xb_residual_layernorm_masked(16, 16, 1, None, None, None, 16, 1, 0, 128, 1e-5, 0, None, 7, None) == 0
    # Fused d128 stack: which shapes split over two workgroups, and the workspace checks.
    # Layout: 256-byte header (timeout counter, finished blocks, generation), 64-bit flags of
    # 128 sequences x layers, K/V slots from a 256-byte boundary.
    slot = 2 * 64 * 128 * 2
    head = lambda layers: (256 + 8 * 128 * layers + 255) // 256 * 256
    assert lib.xb_fused_forward_d128_workspace_bytes(64, 128, 4, 4, 1) == head(4) + 64 * 4 * slot
    assert lib.xb_fused_forward_d128_workspace_bytes(80, 65, 4, 2, 1) == head(2) + 80 * 2 * slot
    for heads in (2, 4, 8, 16):  # up to 128 sequences (one workgroup per CU) at every head_dim <= 64
        assert lib.xb_fused_forward_d128_workspace_bytes(128, 128, heads, 4, 1) == head(4) + 128 * 4 * slot
        assert lib.xb_fused_forward_d128_workspace_bytes(129, 128, heads, 4, 1) == 0
    assert lib.xb_fused_forward_d128_workspace_bytes(64, 64, 4, 4, 1) == 0     # no second half
    assert lib.xb_fused_forward_d128_workspace_bytes(64, 128, 4, 4, 0) == 0    # non-causal
    assert lib.xb_fused_forward_d128_workspace_bytes(64, 128, 1, 4, 1) == 0    # head_dim 128
    need = head(4) + 64 * 4 * slot
    ws_args = (16, 16, 16, 16, 64, 128, 4, 128, 4, -1, None, 1)
    assert lib.xb_fused_forward_d128_ws(*ws_args, 16, need - 1, -1, 0, None) == -7
    assert lib.xb_fused_forward_d128_ws(*ws_args, 24, need, -1, 0, None) == -5
    assert lib.xb_fused_forward_d128_ws(*ws_args, 16, need, -1, 4, None) == -6    # unknown fault flag
    assert lib.xb_fused_forward_d128_ws(16, 16, 16, 16, 64, 129, 4, 128, 4, -1, None, 1, 16, 1 << 30, -1, 0, None) == -4
    assert lib.xb_fused_forward_d128_ws(16, 16, 16, 16, 0, 128, 4, 128, 4, -1, None, 1, None, 0, -1, 0, None) == 0
    # No-allocation decode: a call whose partials exceed the static scratch is refused before any launch
    assert lib.xb_attention_kv_cache_noalloc(16, 16, 16, 16, 20000, 1, 16, 64, 100, 101, 0.1, None) == -9
    assert lib.xb_attention_kv_cache_noalloc(None, 16, 16, 16, 1, 1, 2, 64, 100, 101, 0.1, None) == -1
    assert lib.xb_attention_kv_cache_noalloc(16, 16, 16, 16, 1, 1, 2, 64, 100, 100, 0.1, None) == -2
    _check_noalloc_scratch_rule(lib)
    for code in (0, -1, -2, -3, -4, -5, -6, -7, -8, -9):
        assert lib.xb_strerror(code)
    with pytest.raises(RuntimeError, match="xb_linear failed with code -4"):
        capi.check(-4, "xb_linear")


def test_captured_forwards_run_as_planned(pkg):
    """A captured forward runs its plan's launches on one stream, whatever its form and size."""
    shapes = pkg.OFFICIAL_BENCHMARK_SHAPES
    for shape_id in (1, 6, 8, 11):
        c = shapes[shape_id]
        assert pkg.UserOptimizedTransformer(c).captured_overlap(c.batch_size, c.seq_len) is None
    odd = pkg.UserOptimizedTransformer(pkg.TransformerConfig(7, 64, 1024, 4, 1024, 1, True))
    assert odd.captured_overlap(7, 64, padded=True) is None and odd.captured_overlap(7, 64) is None


def test_stack_forward_argument_checks(capi):
    """xb_stack_forward refuses bad sizes, missing pointers and a small workspace before any launch."""
    import ctypes

    lib = capi.lib()
    need = lib.xb_stack_workspace_bytes(2, 8, 4, 16, 64, -1, -1)
    rows, d = 16, 64
    # residual (FP32), norm, update, then qkv with ctx, in whose place the FFN hidden state goes
    assert need == rows * d * (4 + 2 + 2 + 6 + 2)
    assert lib.xb_stack_workspace_bytes(2, 8, 4, 16, 4096, -1, -1) == rows * (d * 8 + 2 * 4096)
    assert lib.xb_stack_workspace_bytes(2, 8, 4, 16, 64, -1, 100) == \
        need + (lib.xb_attention_kv_cache_workspace_bytes(2, 8, 4, 16, 100) + 255) // 256 * 256
    assert lib.xb_stack_workspace_bytes(2, 8, 0, 16, 64, -1, -1) == -2
    blocks = (capi.XbBlock * 1)()
    stack = capi.XbStack(blocks=blocks, layers=1, heads=4, head_dim=16, ffn_dim=64, causal=1)
    ref = ctypes.addressof(stack)

    def call(x=16, y=16, batch=2, ws=256, ws_bytes=need, valid=None, caches=None, start=0):
        return lib.xb_stack_forward(ref, x, y, valid, batch, 8, -1, -1, -1, -1, -1, caches, start, 8, ws, ws_bytes, None)

    assert call(batch=0) == 0
    assert call(x=None) == -1 and call(y=None) == -1 and call(ws=None) == -1
    assert call(ws_bytes=need - 1) == -7 and call(ws=8) == -5
    assert call(batch=-1) == -2
    assert call(valid=16, caches=16) == -2 and call(caches=16, start=-1) == -2
    stack.layers = 0
    assert call() == -2


def test_row_block_descriptor_reads_nothing_from_the_device(pkg, monkeypatch):
    """Row blocks apply every LayerNorm's affine: their descriptor doesn't ask whether it is (1, 0),
    which takes two reads from the device per LayerNorm, and the per-op one does."""
    import importlib

    kernels = importlib.import_module(pkg.__name__ + ".kernels")
    monkeypatch.setattr(kernels, "pack_linear_fragments", lambda w, out: out.copy_(w.detach().flatten()))
    model = pkg.UserOptimizedTransformer(pkg.TransformerConfig(2, 300, 64, 4, 64, 2, True)).eval()
    asked = []
    monkeypatch.setattr(type(model), "_layer_norm_uses_affine", staticmethod(lambda norm: asked.append(norm) or False))
    stack, blocks, _ = model._native_stack(True)[:3]
    assert not asked and stack.final_affine == blocks[0].norm1_affine == blocks[1].norm2_affine == 1
    stack, blocks, _ = model._native_stack(False)[:3]
    assert len(asked) == 5 and stack.final_affine == blocks[0].norm1_affine == 0
