"""Host-side behaviour of the ComfyUI-facing layer that needs no GPU: state-dict loading rules,
scale bookkeeping, ModelPatcher hooks, LoRA scale slicing, delta reconstruction, Hadamard build."""
import sysconfig
import types

import numpy as np
import pytest
import torch
import torch.nn.utils.parametrize
import torch.nn.utils.prune
from torch.utils._python_dispatch import TorchDispatchMode


@pytest.fixture(autouse=True)
def reset_flags(pkg):
    ops = pkg.Int8TensorwiseOps
    saved = (list(ops.excluded_names), ops.dynamic_quantize, ops.enable_quarot, ops._is_prequantized)
    yield
    ops.excluded_names, ops.dynamic_quantize, ops.enable_quarot, ops._is_prequantized = saved


def load(layer, sd, prefix="blk.0.lin."):
    missing = []
    layer._load_from_state_dict(dict(sd), prefix, {}, True, missing, [], [])
    return missing


def test_prequantized_scalar_scale_becomes_python_float(pkg):
    lin = pkg.Int8TensorwiseOps.Linear(64, 32, bias=True)
    w = torch.randint(-128, 128, (32, 64), dtype=torch.int8)
    sd = {"blk.0.lin.weight": w, "blk.0.lin.weight_scale": torch.tensor(0.0125), "blk.0.lin.bias": torch.zeros(32),
          "blk.0.lin.input_scale": torch.tensor(1.0), "blk.0.lin.comfy_quant": torch.zeros(1)}
    assert load(lin, sd) == []
    assert lin._is_quantized and not lin._is_per_row and lin.weight_scale is None
    assert lin._weight_scale_scalar == pytest.approx(0.0125) and isinstance(lin._get_weight_scale(), float)
    assert lin.weight.dtype == torch.int8 and not lin.weight.requires_grad and torch.equal(lin.weight, w)
    assert lin.weight_comfy_model_dtype == torch.int8 and lin.bias_comfy_model_dtype == torch.float32
    assert pkg.Int8TensorwiseOps._is_prequantized


def test_prequantized_per_row_and_odd_scale_shapes(pkg):
    w = torch.zeros(32, 64, dtype=torch.int8)
    lin = pkg.Int8TensorwiseOps.Linear(64, 32, bias=False)
    load(lin, {"blk.0.lin.weight": w, "blk.0.lin.weight_scale": torch.rand(32, 1).half()})
    assert lin._is_per_row and lin.weight_scale.dtype == torch.float32 and lin.weight_scale.shape == (32, 1)
    assert lin._weight_scale_scalar is None and lin.bias is None
    lin2 = pkg.Int8TensorwiseOps.Linear(64, 32, bias=False)
    load(lin2, {"blk.0.lin.weight": w, "blk.0.lin.weight_scale": torch.rand(32)})   # not [N,1]: kept, treated as one scale
    assert lin2._is_quantized and not lin2._is_per_row and lin2.weight_scale.shape == (32,)
    lin3 = pkg.Int8TensorwiseOps.Linear(64, 32, bias=False)
    load(lin3, {"blk.0.lin.weight": w, "blk.0.lin.weight_scale": 0.5})
    assert lin3._weight_scale_scalar == 0.5


def test_float_weights_stay_float_unless_dynamic_quantize(pkg):
    ops = pkg.Int8TensorwiseOps
    w = torch.randn(32, 64).bfloat16()
    lin = ops.Linear(64, 32, bias=False)
    load(lin, {"blk.0.lin.weight": w})
    assert not lin._is_quantized and lin.weight.dtype == torch.bfloat16
    ops.dynamic_quantize = True
    ops.excluded_names = ["blk.0"]
    lin = ops.Linear(64, 32, bias=False)
    load(lin, {"blk.0.lin.weight": w})
    assert not lin._is_quantized                              # excluded by name
    ops.excluded_names = []
    lin = ops.Linear(64, 1, bias=False)
    load(lin, {"blk.0.lin.weight": torch.randn(1, 64)})
    assert not lin._is_quantized                              # a dimension of 1 is never quantised
    lin = ops.Linear(64, 32, bias=False)
    assert load(lin, {}) == ["blk.0.lin.weight"]              # missing key is reported
    if not torch.cuda.is_available():
        lin = ops.Linear(64, 32, bias=False)
        with pytest.raises(RuntimeError):                      # quantising needs the GPU library: no CPU path
            load(lin, {"blk.0.lin.weight": w})


def test_unquantized_layer_is_a_plain_linear(pkg):
    lin = pkg.Int8TensorwiseOps.Linear(16, 8, bias=True)
    w, b = torch.randn(8, 16), torch.randn(8)
    load(lin, {"blk.0.lin.weight": w, "blk.0.lin.bias": b})
    x = torch.randn(3, 5, 16)
    assert torch.allclose(lin(x), torch.nn.functional.linear(x, w, b))
    assert lin.convert_weight(w) is w


def test_model_patcher_hooks(pkg):
    lin = pkg.Int8TensorwiseOps.Linear(64, 32, bias=True)
    w = torch.randint(-128, 128, (32, 64), dtype=torch.int8)
    load(lin, {"blk.0.lin.weight": w, "blk.0.lin.weight_scale": torch.rand(32, 1), "blk.0.lin.bias": torch.zeros(32)})
    assert lin.convert_weight(torch.zeros(1)) is lin.weight               # int8 payload handed to the adapter
    w2 = torch.randint(-128, 128, (32, 64), dtype=torch.int8)
    assert lin.set_weight(w2, return_weight=True) is w2
    lin.set_weight(w2)
    assert torch.equal(lin.weight, w2) and isinstance(lin.weight, torch.nn.Parameter)
    w3 = torch.randint(-128, 128, (32, 64), dtype=torch.int8)
    keep = lin.weight
    lin.set_weight(w3, inplace_update=True)
    assert lin.weight is keep and torch.equal(lin.weight, w3)
    assert lin.set_bias(None) is None
    nb = torch.ones(32)
    lin.set_bias(nb)
    assert torch.equal(lin.bias, nb)
    lin.set_bias(torch.full((32,), 2.0), inplace_update=True)
    assert float(lin.bias[0]) == 2.0


def test_pass_through_layers_and_conv_nd(pkg):
    ops = pkg.Int8TensorwiseOps
    assert isinstance(ops.conv_nd(2, 3, 4, 3), ops.Conv2d) and isinstance(ops.conv_nd(3, 3, 4, 3), ops.Conv3d)
    with pytest.raises(ValueError):
        ops.conv_nd(1, 3, 4, 3)
    for name in ("GroupNorm", "LayerNorm", "ConvTranspose2d", "Embedding"):
        assert hasattr(ops, name)
    assert ops.use_triton is True and ops.excluded_names == []


def test_scale_slicing_rules_of_both_adapters(pkg):
    ws = torch.arange(96, dtype=torch.float32).reshape(96, 1)
    single = pkg.INT8LoRAPatchAdapter(set(), (None,) * 6, ws, seed=1)
    assert single._get_effective_scale(torch.zeros(32, 8), (0, 32, 32)).flatten().tolist() == list(range(32, 64))
    assert single._get_effective_scale(torch.zeros(96, 8), (0, 32, 32)).shape == (32, 1)   # offset wins even if rows match
    assert single._get_effective_scale(torch.zeros(32, 8), None).flatten().tolist() == list(range(32))
    assert single._get_effective_scale(torch.zeros(96, 8), None) is ws
    assert single._get_effective_scale(torch.zeros(32, 8), (0, 80, 32)).shape == (16, 1)   # clipped at the end
    assert pkg.INT8LoRAPatchAdapter(set(), (None,) * 6, 0.5)._get_effective_scale(torch.zeros(4, 4), (0, 1, 2)) == 0.5
    inner = pkg.INT8LoRAPatchAdapter({"k"}, (None,) * 6, ws)
    merged = pkg.INT8MergedLoRAPatchAdapter([(inner, 1.0)], ws, seed=2)
    assert merged.loaded_keys == {"k"} and merged.seed == 2
    assert merged._get_effective_scale(torch.zeros(32, 8), (0, 32, 32)).flatten().tolist() == list(range(32, 64))
    assert merged._get_effective_scale(torch.zeros(96, 8), (0, 32, 32)) is ws              # older rule: only on mismatch
    assert merged._get_effective_scale(torch.zeros(32, 8), (1, 0, 8)).flatten().tolist() == list(range(32))


def test_reconstruct_lora_diff_variants(pkg):
    f = pkg.int8_quant.reconstruct_lora_diff
    g = torch.Generator().manual_seed(0)
    up, down = torch.randn(12, 4, generator=g), torch.randn(4, 10, generator=g)
    d, s = f((up, down, 8.0, None, None, None), (12, 10), "cpu", torch.float32, 0.5)
    assert torch.allclose(d, up @ down) and s == pytest.approx(8.0 / 4 * 0.5)
    mid = torch.randn(4, 4, generator=g)
    d, s = f((up, down, None, mid, None, None), (12, 10), "cpu", torch.float32, 0.7)
    assert torch.allclose(d, up @ mid @ down, atol=1e-5) and s == 0.7
    w1a, w1b, w2a, w2b = (torch.randn(*sh, generator=g) for sh in [(12, 3), (3, 10), (12, 3), (3, 10)])
    d, s = f((w1a, w1b, 3.0, w2a, w2b, None, None, None), (12, 10), "cpu", torch.float32, 1.0)
    assert torch.allclose(d, (w1a @ w1b) * (w2a @ w2b)) and s == pytest.approx(1.0)
    k1, k2 = torch.randn(3, 2, generator=g), torch.randn(4, 5, generator=g)
    d, s = f((k1, k2, 1.0, None, None, None, None, None, None), (12, 10), "cpu", torch.float32, 2.0)
    assert torch.allclose(d, torch.kron(k1, k2)) and s == 2.0
    assert f((1, 2, 3), (1,), "cpu", torch.float32, 1.0) == (None, 1.0)


def test_build_hadamard(pkg):
    from scipy.linalg import hadamard

    H = pkg.quarot.build_hadamard(128)
    assert np.array_equal(H.numpy(), (torch.tensor(hadamard(128), dtype=torch.float32) / (128**0.5)).numpy())
    assert torch.allclose(H @ H.T, torch.eye(128), atol=1e-6) and torch.equal(H, H.T)
    assert pkg.quarot.build_hadamard(128) is H                         # cached
    Hb = pkg.quarot.build_hadamard(128, dtype=torch.bfloat16)
    assert Hb.dtype == torch.bfloat16 and float(Hb[0, 0]) == 0.08837890625
    with pytest.raises(ValueError):
        pkg.quarot.build_hadamard(96)
    with pytest.raises(ValueError):
        pkg.quarot.rotate_weight(torch.zeros(4, 100))
    with pytest.raises(ValueError):
        pkg.quarot.rotate_activation(torch.zeros(4, 256), None, 64)


def test_quantize_int8_given_scale_and_dequantize(pkg):
    x = torch.tensor([[0.5, -1.26, 100.0, -100.0, 0.024, 0.026]])
    q = pkg.quantize_int8(x, 0.05)
    assert q.tolist() == [[10, -25, 127, -128, 0, 1]]
    assert torch.allclose(pkg.dequantize(q, 0.05), torch.tensor([[0.5, -1.25, 6.35, -6.4, 0.0, 0.05]]))


def test_aliases_keep_the_reference_names(pkg):
    assert pkg.triton_quantize_rowwise is pkg.hip_quantize_rowwise
    assert pkg.triton_int8_linear is pkg.hip_int8_linear
    assert pkg.triton_int8_linear_per_row is pkg.hip_int8_linear_per_row
    with pytest.raises(ValueError):
        pkg.quantize_int8_axiswise(torch.zeros(4, 8), dim=0)


class _Host:
    """Stands in for the native host module: notes its arguments and leaves every call to the general path."""

    def __init__(self):
        self.calls = []

    def linear(self, *args):
        self.calls.append(args)


@pytest.fixture
def host(pkg, monkeypatch):
    h = _Host()
    monkeypatch.setattr(pkg._lib, "host", lambda: h)
    return h


def native(pkg, lin, x, **kw):
    a = dict(prologue=pkg._lib.PRO_NONE, mod_scale=None, mod_shift=None, eps=1e-6, gate=None, residual=None, norm_weight=None, fused_add=False)
    return lin._forward_native(x, **{**a, **kw})


@pytest.mark.parametrize("kept_as", ["parameter", "none", "buffer", "attribute", "parametrised"])
def test_native_host_path_never_drops_a_bias(pkg, host, kept_as):
    """What the layer's bias attribute gives is what the native path is handed, or the call is left to the general path."""
    lin = pkg.Int8TensorwiseOps.Linear(64, 32, bias=True)
    load(lin, {"blk.0.lin.weight": torch.ones(32, 64, dtype=torch.int8), "blk.0.lin.weight_scale": torch.tensor(0.5),
               "blk.0.lin.bias": torch.arange(32.0)})
    if kept_as == "none":
        lin.bias = None
    elif kept_as == "buffer":
        del lin.bias
        lin.register_buffer("bias", torch.arange(32.0))
    elif kept_as == "attribute":
        torch.nn.utils.prune.identity(lin, "bias")
    elif kept_as == "parametrised":
        torch.nn.utils.parametrize.register_parametrization(lin, "bias", torch.nn.Identity())
    assert (lin.bias is None) == (kept_as == "none")
    assert native(pkg, lin, torch.zeros(20, 64, dtype=torch.bfloat16)) is None
    if kept_as in ("parameter", "none"):
        assert len(host.calls) == 1
    for args in host.calls:
        assert args[3] is lin.bias


def stack(pkg, pairs, n=48, k=64):
    """A stack adapter of (up, down) pairs with the strengths 1, 1/2, 1/4, ..., and an int8 weight for it."""
    parts = [(pkg.INT8LoRAPatchAdapter({"k"}, (u, d, None, None, None, None), 0.01), 0.5**i) for i, (u, d) in enumerate(pairs)]
    return pkg.INT8MergedLoRAPatchAdapter(parts, 0.01, seed=3), torch.zeros(n, k, dtype=torch.int8)


def test_stacked_factors_of_loras_that_require_grad(pkg):
    """LoRA factors that are parameters are stacked like any others."""
    g = torch.Generator().manual_seed(5)
    pairs = [(torch.nn.Parameter(torch.randn(48, r, generator=g)), torch.nn.Parameter(torch.randn(r, 64, generator=g))) for r in (4, 8)]
    adapter, w = stack(pkg, pairs)
    up, down = adapter._stacked_factors(w, torch.device("cpu"))
    assert not up.requires_grad and not down.requires_grad
    assert torch.equal(up, torch.cat([u.detach() for u, _ in pairs], 1))
    assert torch.equal(down, torch.cat([d.detach() * 0.5**i for i, (_, d) in enumerate(pairs)]))


def test_stacked_factors_refuses_a_lora_whose_factors_disagree_on_the_rank(pkg):
    """Ranks that mismatch crosswise add up to the same total; such a stack is left to the general path, whose product
    raises."""
    adapter, w = stack(pkg, [(torch.ones(48, 16), torch.ones(32, 64)), (torch.ones(48, 32), torch.ones(16, 64))])
    assert adapter._stacked_factors(w, torch.device("cpu")) is None
    with pytest.raises(RuntimeError):
        adapter.calculate_weight(torch.zeros(48, 64), "k", 1.0, 1.0, None, None)


def test_stacked_factors_leaves_empty_loras_to_the_general_path(pkg):
    """A stack of nothing but LoRAs of rank 0 has a delta of zeros, which the fused kernel has no form for."""
    adapter, w = stack(pkg, [(torch.ones(48, 0), torch.ones(0, 64))] * 2)
    assert adapter._stacked_factors(w, torch.device("cpu")) is None
    adapter, w = stack(pkg, [(torch.ones(48, 0), torch.ones(0, 64)), (torch.ones(48, 4), torch.ones(4, 64))])
    assert adapter._stacked_factors(w, torch.device("cpu"))[0].shape == (48, 4)


class Conversions(TorchDispatchMode):
    def __init__(self):
        super().__init__()
        self.count = 0

    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        self.count += func is torch.ops.aten._to_copy.default
        return func(*args, **(kwargs or {}))


@pytest.mark.parametrize("count,rotated", [(1, False), (1, True), (2, False), (2, True), (9, False), (9, True)])
def test_a_merge_that_draws_no_noise_itself_prepares_its_operands_once(pkg, monkeypatch, count, rotated):
    """Whichever route a stack takes in the end, every factor is moved and widened once and one generator is seeded; and so
    for a single LoRA."""
    monkeypatch.setattr(pkg.int8_quant, "compute_device", lambda: torch.device("cpu"))
    monkeypatch.setattr(pkg.Int8TensorwiseOps, "enable_quarot", rotated)
    monkeypatch.setattr(pkg._lib, "rotate128", lambda t: t)
    monkeypatch.setattr(pkg._lib, "lora_merge_sr_drawn", lambda *a: None)
    merges, seeds, seeded = [], [], pkg.int8_quant._seeded
    monkeypatch.setattr(pkg.int8_quant, "_seeded", lambda *a: seeds.append(a) or seeded(*a))
    monkeypatch.setattr(pkg._lib, "lora_merge_sr", lambda w, scale, noise, **k: merges.append((noise, k)) or w)
    g = torch.Generator().manual_seed(6)
    pairs = [(torch.randn(48, 4, generator=g).half(), torch.randn(4, 128, generator=g).half()) for _ in range(count)]
    stacked, w = stack(pkg, pairs, k=128)
    for adapter in (stacked, stacked.patches[0][0]):
        loras, seed = len(getattr(adapter, "patches", [0])), adapter.seed
        with Conversions() as conversions:
            adapter.calculate_weight(w, "k", 1.0, 1.0, None, None)
        assert conversions.count == 2 * loras and len(seeds) == 1
        noise, operands = merges[0]
        assert torch.equal(noise, torch.rand(48, 128, generator=torch.Generator().manual_seed(seed)))
        assert torch.equal(operands["up"], torch.cat([u.float() for u, _ in pairs[:loras]], 1))
        merges.clear(), seeds.clear()


@pytest.mark.parametrize("rows,k", [(4, 12288), (16, 10240), (17, 12288), (40, 12288), (40, 10224)])
def test_native_host_path_takes_no_workspace_before_the_call_is_decided(pkg, host, monkeypatch, rows, k):
    """The memory of the K split is asked for by the native function itself, behind its checks: a call that it does not take,
    or one of 16 rows or fewer, costs none."""
    asked = []
    monkeypatch.setattr(pkg._lib, "_splitk_workspace", lambda *a: asked.append(a))
    lin = pkg.Int8TensorwiseOps.Linear(k, 8, bias=False)
    load(lin, {"blk.0.lin.weight": torch.ones(8, k, dtype=torch.int8), "blk.0.lin.weight_scale": torch.tensor(0.5)})
    assert native(pkg, lin, torch.zeros(rows, k, dtype=torch.bfloat16)) is None
    assert asked == [] and (host.calls[0][16] is None) == (k < pkg._lib.SPLITK_MIN_K)


def test_host_extension_of_another_torch_or_python_is_not_loaded(pkg, monkeypatch):
    """The extension is compiled against one torch and one Python: with others it is missing, and the error says what to do."""
    L = pkg._lib
    assert L.host() is L.host()
    for place, name, value in ((torch, "__version__", "0.0.1+other"), (sysconfig, "get_config_var", lambda key: "cpython-00")):
        with monkeypatch.context() as m:
            m.setattr(L, "_host", None)
            m.setattr(place, name, value)
            with pytest.raises(RuntimeError, match="build.py"):
                L.host()


@pytest.mark.parametrize("flag", [True, 1, np.bool_(True), False, 0])
def test_native_host_path_is_told_the_scale_mode_as_a_truth_value(pkg, host, flag):
    """Per-row scales marked by anything true are per-row scales, as in the general path."""
    lin = pkg.Int8TensorwiseOps.Linear(64, 32, bias=False)
    load(lin, {"blk.0.lin.weight": torch.ones(32, 64, dtype=torch.int8), "blk.0.lin.weight_scale": torch.rand(32, 1)})
    lin._is_per_row = flag
    native(pkg, lin, torch.zeros(20, 64, dtype=torch.bfloat16))
    assert host.calls[0][4] is bool(flag)


def test_a_lora_without_a_native_form_does_not_ask_for_one(pkg, monkeypatch):
    """Rank, rows and width tell it before anything is prepared for the native path; what they let through reaches it."""
    lin = pkg.Int8TensorwiseOps.Linear(64, 48, bias=False, dtype=torch.bfloat16)
    lin.weight = torch.nn.Parameter(torch.zeros(48, 64, dtype=torch.int8), requires_grad=False)
    lin._is_quantized, lin._weight_scale_scalar = True, 0.01
    asked = []
    monkeypatch.setattr(pkg._lib, "host", lambda: types.SimpleNamespace(linear_lora=lambda *a: asked.append(a)))

    def call(rank, rows, lora_b=True, rotated=False, width=64, **other):
        lin.lora_A = torch.zeros(rank, width, dtype=torch.bfloat16)
        lin.lora_B = torch.zeros(48, rank, dtype=torch.bfloat16) if lora_b else None
        lin._use_quarot = rotated
        del asked[:]
        args = dict(prologue=pkg._lib.PRO_NONE, mod_scale=None, mod_shift=None, eps=1e-6, gate=None, residual=None, norm_weight=None, fused_add=False)
        assert lin._forward_native(torch.zeros(rows, width, dtype=torch.bfloat16), **{**args, **other}) is None
        return len(asked)

    assert call(16, 17) == 1 and call(64, 17) == 1
    assert call(8, 40) == 0 and call(16, 16) == 0 and call(16, 40, lora_b=False) == 0 and call(16, 40, rotated=True) == 0
    assert call(16, 40, width=6272) == 0 and call(16, 40, gate=torch.zeros(48)) == 0 and call(16, 40, residual=torch.zeros(40, 48)) == 0
    assert call(16, 40, prologue=pkg._lib.PRO_GELU_TANH) == 0
