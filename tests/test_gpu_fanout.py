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


@pytest.mark.gpu
@pytest.mark.parametrize("widths", [(3456, 256, 256), (256, 3456), (256, 256)])
def test_narrow_layers_keep_their_k_split_beside_wide_ones(pkg, L, dev, widths, monkeypatch):
    """Eager, on a stream of its own and captured: the partial sums show that the layers of 256 columns were split (135 tiles of
    128 x 128, those of 3456, are more than a split takes)."""
    rows, K = 520, 10240
    lins = layers_of(pkg, dev, widths, K, torch.bfloat16)
    x = torch.randn(rows, K, device=dev).bfloat16()
    want = [lin(x) for lin in lins]
    handed, ask = [], L._splitk_workspace
    monkeypatch.setattr(L, "_splitk_workspace", lambda *a: handed.append(ask(*a)) or handed[-1])
    untouched = 0x5a5a5a5a   # (no sum of 10240 products)

    def partials(work):
        return work[L._SPLITK_COUNTER_BYTES:].view(torch.int32)

    def check(outs):
        torch.cuda.synchronize()
        assert all(torch.equal(o, v) for o, v in zip(outs, want))
        written = int((partials(handed[-1]) != untouched).sum())
        assert written >= 520 * 256 and int(handed[-1][:L._SPLITK_COUNTER_BYTES].sum()) == 0

    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    for stream in (torch.cuda.current_stream(), side):
        with torch.cuda.stream(stream):
            partials(ask(x, rows, 256, K)).fill_(untouched)
            check(pkg.forward_fanout(lins, x))
    assert len(handed) == 2 and handed[0].data_ptr() != handed[1].data_ptr()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        outs = pkg.forward_fanout(lins, x)
    assert len(handed) == 3 and all(handed[2].data_ptr() != h.data_ptr() for h in handed[:2])
    for _ in range(3):
        partials(handed[2]).fill_(untouched)
        for o in outs:
            o.zero_()
        graph.replay()
        check(outs)
        assert all(torch.equal(o, v) for o, v in zip(pkg.forward_fanout(lins, x), want))   # an eager call in between
        handed.pop()


@pytest.mark.gpu
@pytest.mark.parametrize("rows,K,widths,dtype,opts,reason", [
    (300, 512, (1536, 1536, 1536), torch.bfloat16, {}, "patched"), (4096, 256, (3840, 3840, 3840), torch.float16, {"rotate": True}, "patched"),
    (40, 256, (64,) * 9, torch.bfloat16, {}, "count"), (33, 384, (64, 64, 192, 8, 8, 8, 8, 192, 100), torch.float16, {}, "count"),
    (100, 384, (96, 192, 192, 8), torch.bfloat16, {"per_row": (False, True, True, True), "bias": (True, False, True, True)}, "patched"),
    (70, 256, (128, 128, 128), torch.float16, {"per_row": (False, True, False)}, "patched"), (520, 10240, (3456, 256, 256), torch.bfloat16, {}, "patched"),
    (50, 200, (100, 100), torch.bfloat16, {}, "patched"), (64, 256, (128, 128), torch.bfloat16, {}, "bias"),
])
def test_the_general_path_of_the_fanout_is_the_layers_own_forward(pkg, L, dev, rows, K, widths, dtype, opts, reason, monkeypatch):
    """What the native call leaves: more layers than it takes, a bias of another type behind one launch's, and, to have every
    form here, calls that it would take."""
    lins = layers_of(pkg, dev, widths, K, dtype, **opts)
    if reason == "bias":
        lins[1].bias = torch.nn.Parameter(lins[1].bias.float(), requires_grad=False)
    if reason in ("patched", "bias"):
        monkeypatch.setattr(pkg.int8_quant, "_fanout_native", lambda *a: None)
    look, looked = L._i8_matrix, []
    monkeypatch.setattr(L, "_i8_matrix", lambda *a: looked.append(a[1]) or look(*a))
    x = torch.randn(1, rows, K, device=dev).to(dtype)
    scale, shift, weight = (torch.randn(K, device=dev).to(dtype) * 0.2 for _ in range(3))
    calls = [{}, {"prologue": L.PRO_MODULATE, "mod_scale": scale, "mod_shift": shift}]
    if K % 16 == 0:
        calls += [{"prologue": L.PRO_RMS_NORM, "norm_weight": weight, "mod_scale": scale, "eps": 1e-5}]
    for t in (x, x[0]):
        for kw in calls:
            looked.clear()
            outs = pkg.forward_fanout(lins, t, **kw)
            assert looked == ["a", "w"] * len(lins)   # (every layer's operands once)
            assert all(torch.equal(o, lin(t, **kw)) for o, lin in zip(outs, lins)) and len(outs) == len(lins)
