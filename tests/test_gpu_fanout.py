"""Several layers on one quantisation through the native host path: which calls take it, and the layers' own bits."""
import pytest
import torch


def layers_of(pkg, dev, widths, K, dtype, rotate=False, per_row=None, bias=None):
    out = []
    for i, n in enumerate(widths):
        g = torch.Generator(device=dev).manual_seed(100 * i + n)
        lin = pkg.Int8TensorwiseOps.Linear(K, n, bias=bias is None or bias[i], device="meta")
        row = per_row is None or per_row[i]
        state = {"weight": torch.randint(-127, 128, (n, K), dtype=torch.int8, generator=g, device=dev),
                 "weight_scale": torch.rand(n, 1, generator=g, device=dev) * 0.002 + 1e-3 if row else torch.tensor(0.002)}
        if bias is None or bias[i]:
            state["bias"] = torch.randn(n, generator=g, device=dev).to(dtype)
        lin._load_from_state_dict(state, "", {}, True, [], [], [])
        lin._use_quarot = rotate
        out.append(lin)
    return out


@pytest.mark.gpu
@pytest.mark.parametrize("rows,K,widths,dtype,opts", [
    (300, 512, (1536, 1536, 1536), torch.bfloat16, {}), (4096, 256, (3840, 3840, 3840), torch.float16, {"rotate": True}),   # one launch
    (70, 256, (128,) * 5, torch.bfloat16, {}), (33, 256, (64,) * 8, torch.float16, {}),                                     # more than a launch takes
    (100, 384, (96, 192, 192, 8), torch.bfloat16, {"per_row": (False, True, True, True), "bias": (True, False, True, True)}),
    (17, 10240, (256, 256), torch.bfloat16, {}), (520, 12288, (3072, 3072), torch.float16, {}),                             # K split
    (50, 200, (100, 100), torch.bfloat16, {}), (90, 128, (1, 3, 3), torch.float16, {}),                                     # widths that fit no tile
])
def test_fanout_is_the_layers_own_forward(pkg, L, dev, rows, K, widths, dtype, opts, monkeypatch):
    lins = layers_of(pkg, dev, widths, K, dtype, **opts)
    x = torch.randn(1, rows, K, device=dev).to(dtype)
    scale, shift, weight = (torch.randn(K, device=dev).to(dtype) * 0.2 for _ in range(3))
    calls = [{}, {"prologue": L.PRO_GELU_TANH}, {"prologue": L.PRO_MODULATE, "mod_scale": scale, "mod_shift": shift}]
    if K % 16 == 0:
        calls += [{"prologue": L.PRO_RMS_NORM, "norm_weight": weight, "mod_scale": scale, "eps": 1e-5},
                  {"prologue": L.PRO_NORM_MODULATE, "mod_scale": scale, "mod_shift": shift, "fused_add": True}]
    native = pkg.int8_quant._fanout_native
    taken = []
    monkeypatch.setattr(pkg.int8_quant, "_fanout_native", lambda *a: taken.append(native(*a)) or taken[-1])
    strided = torch.randn(1, rows, 2 * K, device=dev).to(dtype)[..., :K]   # rows apart
    for t in (x, x[0], strided):
        for kw in calls:
            outs = pkg.forward_fanout(lins, t, **kw)
            assert all(torch.equal(o, lin(t, **kw)) for o, lin in zip(outs, lins)) and len(outs) == len(lins)
    assert all(o is not None for o in taken[:len(calls)])


@pytest.mark.gpu
def test_calls_that_the_native_fanout_leaves_to_the_general_path(pkg, L, dev):
    lins = layers_of(pkg, dev, (64, 64), 256, torch.bfloat16)
    native = lambda ls, x, **kw: pkg.int8_quant._fanout_native(ls, x, False, kw.get("prologue", L.PRO_NONE), kw.get("mod_scale"), None, 1e-6, None, False)
    x = torch.randn(40, 256, device=dev).bfloat16()
    assert native(lins, x) is not None
    assert native(lins, x[:16]) is None and native(lins, x[0]) is None and native(lins, x.float()) is None and native(lins, x[:, ::2]) is None
    assert native(lins * 5, x) is None and native(lins, x.cpu()) is None
    assert native(lins, x, prologue=L.PRO_SILU_GATE, mod_scale=x[:20]) is None and native(lins, x, prologue=99) is None
    other = layers_of(pkg, dev, (64,), 128, torch.bfloat16)
    assert native([lins[0], other[0]], x) is None
    lins[1].comfy_cast_weights = True
    assert native(lins, x) is None
    lins[1].comfy_cast_weights, lins[1]._use_quarot = False, True
    assert native(lins, x) is None
    lins[1]._use_quarot, lins[1].lora_A = False, torch.randn(16, 256, device=dev).bfloat16()
    assert native(lins, x) is None
