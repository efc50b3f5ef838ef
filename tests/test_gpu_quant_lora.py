"""The quantiser that forms a dynamic LoRA's first product in the same launch, and the layer that runs it.  The reference
adds x @ lora_A.T @ lora_B.T to the layer's result (reference int8_quant.py:741-744,768)."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu


def quant_lora(L, x, a):
    M, K = x.shape
    q = torch.empty(M, K, dtype=torch.int8, device=x.device)
    scale = torch.empty(M, 1, device=x.device)
    t = torch.empty(M, a.shape[0], dtype=x.dtype, device=x.device)
    fn = L.lib().i8f_internal_quant_lora
    fn.argtypes = [ctypes.c_void_p, ctypes.c_int] + [ctypes.c_int64] * 3 + [ctypes.c_void_p, ctypes.c_int64] + [ctypes.c_void_p] * 4
    rc = fn(x.data_ptr(), L.dtype_code(x.dtype), M, K, x.stride(0), a.data_ptr(), a.shape[0], q.data_ptr(), scale.data_ptr(), t.data_ptr(),
            L._stream(x))
    return rc, q, scale, t


@pytest.mark.parametrize("M,K,rank,dtype,pad", [
    (1, 64, 16, torch.bfloat16, 0),        # one block: seven waves have none
    (17, 576, 32, torch.float16, 8),       # a second block for one wave only, rows at a stride
    (15, 1088, 48, torch.bfloat16, 0),     # 17 blocks, no full row tile
    (33, 2048, 64, torch.float16, 64),
    (16, 3072, 32, torch.bfloat16, 0),
    (1357, 3072, 64, torch.bfloat16, 0),
    (31, 4096, 48, torch.float16, 0),
    (9, 4160, 32, torch.bfloat16, 0),      # 65 blocks: a ninth for one wave
    (40, 6144, 16, torch.float16, 0),
])
def test_same_bytes_as_the_quantiser_and_the_product_in_32_bits(L, M, K, rank, dtype, pad):
    gen = torch.Generator(device="cuda").manual_seed(M * 31 + K)
    x = torch.randn(M, K + pad, device="cuda", generator=gen).to(dtype)[:, :K]
    x[:, 3] *= 30.0
    x[M // 2] = 0
    a = (torch.randn(rank, K, device="cuda", generator=gen) * 0.02).to(dtype)
    rc, q, scale, t = quant_lora(L, x, a)
    assert rc == 0
    want_q, want_scale = L.quant_rowwise(x)
    assert torch.equal(q, want_q) and torch.equal(scale, want_scale.view(-1, 1))
    exact = x.double() @ a.double().t()
    # one rounding of the result, and K binary32 additions (products of 16-bit values are exact)
    half_ulp = 2.0 ** -9 if dtype == torch.bfloat16 else 2.0 ** -12
    bound = 2 * half_ulp * exact.abs() + K * 2.0 ** -23 * (x.double().abs() @ a.double().abs().t()) + 2.0 ** -24
    assert bool(((t.double() - exact).abs() <= bound).all())


def test_values_that_are_not_finite_stay_in_their_row(L):
    x = torch.randn(40, 1152, device="cuda").to(torch.bfloat16)
    x[3, 7], x[20, 1100], x[21] = float("inf"), float("nan"), float("nan")
    a = (torch.randn(32, 1152, device="cuda") * 0.02).to(torch.bfloat16)
    a[5, 1] = float("inf")
    _, q, scale, t = quant_lora(L, x, a)
    want_q, want_scale = L.quant_rowwise(x)
    assert torch.equal(q, want_q) and torch.equal(scale.view(-1).view(torch.int32), want_scale.view(-1).view(torch.int32))
    assert torch.equal(t.isnan(), (x.float() @ a.float().t()).isnan()) and torch.equal(t.isinf(), (x.float() @ a.float().t()).isinf())


@pytest.mark.parametrize("M,K,rank", [(64, 64 * 97, 16), (64, 4160, 48), (64, 100, 16), (64, 128, 8), (64, 128, 80), (0, 128, 16)])
def test_refused(L, M, K, rank):
    x = torch.zeros(max(M, 1), K, device="cuda", dtype=torch.bfloat16)[:M]
    assert quant_lora(L, x, torch.zeros(rank, K, device="cuda", dtype=torch.bfloat16))[0] != 0


def layer_with_a_lora(pkg, K, N, rank, dtype, alpha=None, per_row=False, bias=True):
    lin = pkg.Int8TensorwiseOps.Linear(K, N, bias=bias, device="cuda", dtype=dtype)
    lin.weight = torch.nn.Parameter(torch.randint(-127, 128, (N, K), dtype=torch.int8, device="cuda"), requires_grad=False)
    if bias:
        lin.bias = torch.nn.Parameter(torch.randn(N, device="cuda", dtype=dtype), requires_grad=False)
    lin._is_quantized, lin._is_per_row = True, per_row
    scale = torch.rand(N, 1, device="cuda") * 1e-3 + 1e-4 if per_row else torch.tensor(7e-4, device="cuda")
    lin._weight_scale_scalar = None
    lin.register_buffer("weight_scale", scale)
    lin.lora_A = (torch.randn(rank, K, device="cuda") * 0.02).to(dtype)
    lin.lora_B = (torch.randn(N, rank, device="cuda") * 0.1).to(dtype)
    lin.lora_alpha = alpha
    return lin


def native(pkg, lin, x):
    return lin._forward_native(x, pkg._lib.PRO_NONE, None, None, 1e-6, None, None, None, False)


def check_against_general(lin, x, y, monkeypatch):
    K, N = x.shape[-1], lin.weight.shape[0]
    with monkeypatch.context() as m:
        m.setattr(type(lin), "_forward_native", lambda self, *a: None)
        general = lin(x)
    assert y.shape == general.shape and y.dtype == general.dtype
    # t may round to a neighbour in a few places (another order of its binary32 sums): one unit of it through |lora_B|, then the
    # roundings of side, its product with alpha and the sum
    t = (x.reshape(-1, K).float() @ lin.lora_A.float().t()).abs()
    side = (t @ lin.lora_B.float().abs().t()) * (1.0 if lin.lora_alpha is None else lin.lora_alpha)
    bound = (side * 2.0 ** -7 + general.reshape(-1, N).float().abs() * 2.0 ** -7).view_as(general)
    assert bool(((y.float() - general.float()).abs() <= bound).all())


@pytest.mark.parametrize("shape,N,rank,alpha,per_row,bias,dtype,pad,taken", [
    ((17, 256), 136, 16, None, False, True, torch.bfloat16, 0, True),
    ((2, 100, 1536), 520, 32, 0.7, True, True, torch.bfloat16, 0, True),
    ((333, 4096), 1024, 64, 2, True, False, torch.bfloat16, 0, True),
    ((3, 61, 1152), 264, 48, 1.5, True, True, torch.float16, 128, True),      # rows at a stride
    ((97, 6144), 136, 32, None, False, True, torch.float16, 0, True),         # the widest rows
    ((16384, 256), 136, 16, None, True, True, torch.bfloat16, 0, True),       # the most rows
    ((300, 4224), 264, 64, None, False, True, torch.bfloat16, 0, False),      # no room for that rank at this width: the general path
    ((97, 6272), 136, 32, None, False, True, torch.bfloat16, 0, False),
    ((50, 1536), 256, 24, 0.5, False, True, torch.bfloat16, 0, False),        # a rank between two steps
    ((16385, 256), 136, 16, None, True, True, torch.bfloat16, 0, False),
    ((16, 256), 136, 16, None, True, True, torch.bfloat16, 0, False),         # the small-batch form
    ((33, 256), 136, 16, None, True, True, torch.bfloat16, 4, False),         # rows that are not aligned
])
def test_layer_with_a_lora(pkg, shape, N, rank, alpha, per_row, bias, dtype, pad, taken, monkeypatch):
    torch.manual_seed(N)
    K = shape[-1]
    lin = layer_with_a_lora(pkg, K, N, rank, dtype, alpha, per_row, bias)
    x = torch.randn(*shape[:-1], K + pad, device="cuda").to(dtype)[..., :K]
    y = native(pkg, lin, x)
    assert (y is not None) == taken
    if taken:
        assert torch.equal(y, lin(x))
        check_against_general(lin, x, y, monkeypatch)


def test_layer_with_a_lora_under_autocast_is_the_general_paths(pkg, monkeypatch):
    torch.manual_seed(1)
    lin = layer_with_a_lora(pkg, 512, 136, 16, torch.bfloat16)
    x = torch.randn(40, 512, device="cuda").to(torch.bfloat16)
    assert native(pkg, lin, x) is not None
    with torch.autocast("cuda", dtype=torch.float16):
        assert native(pkg, lin, x) is None


def test_layer_with_a_lora_on_another_stream(pkg, monkeypatch):
    torch.manual_seed(2)
    lin = layer_with_a_lora(pkg, 3072, 1024, 32, torch.bfloat16)
    x = torch.randn(1357, 3072, device="cuda").to(torch.bfloat16)
    want = native(pkg, lin, x)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        late = x.roll(1, 0)   # made on the stream that uses it, behind work that takes longer than the launches
        for _ in range(20):
            late = late.roll(1, 0)
        got = native(pkg, lin, late)
        back = got.roll(-21, 0)
    side.synchronize()
    assert torch.equal(back, want)
