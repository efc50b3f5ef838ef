"""The gated residual where the pieces of a gate are shared by the passes of a wave and where they are not: rows per gate that
end inside a wave's tile, tiles whose passes repeat their columns every time (128 columns) or every third time (96), ragged edges."""
import pytest
import torch


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,rows_per_gate,dtype", [
    (4032, 3072, 128, 4032, torch.bfloat16), (4032, 3072, 128, 96, torch.bfloat16), (4000, 3064, 256, 40, torch.float16),  # 256 x 192
    (4608, 3072, 128, 4608, torch.bfloat16), (4608, 3072, 128, 288, torch.float16), (4600, 3064, 128, 8, torch.bfloat16),  # 256 x 256
    (512, 3072, 12288, 512, torch.bfloat16), (510, 3064, 12288, 85, torch.bfloat16),                                       # 128 x 96, K split
    (500, 9208, 256, 50, torch.float16), (100, 1000, 128, 25, torch.float32), (650, 6144, 128, 130, torch.bfloat16),
])
def test_gated_residual_equals_the_tensor_operations(L, dev, M, N, K, rows_per_gate, dtype):
    g = torch.Generator(device=dev).manual_seed(M + N)
    x, scale = L.quant_rowwise(torch.randn(M, K, generator=g, device=dev))
    w, ws = L.quant_rowwise(torch.randn(N, K, generator=g, device=dev) * 0.02)
    gate = torch.randn(M // rows_per_gate, N, generator=g, device=dev).to(dtype)
    residual = torch.randn(M, N, generator=g, device=dev).to(dtype)
    plain = L.linear_w8a8(x, scale, w, ws, None, dtype, L.EPI_TORCH)
    got = L.linear_w8a8(x, scale, w, ws, None, dtype, L.EPI_TORCH, addend=residual, gate=gate)
    assert torch.equal(got, residual + gate.repeat_interleave(rows_per_gate, 0) * plain)


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,rows_per_gate,dtype", [
    (4600, 3064, 128, 4600, torch.bfloat16), (4600, 3064, 128, 46, torch.float16),   # 256 x 256
    (4000, 3064, 256, 4000, torch.float16), (600, 1000, 128, 200, torch.float32), (17, 40, 128, 1, torch.bfloat16),
    (510, 3064, 12288, 85, torch.bfloat16),                                          # 128 x 96, K split
])
@pytest.mark.parametrize("absent", ["gate", "residual", "neither"])
def test_absent_operands_signed_zeros_infinities_and_the_residual_as_output(L, dev, M, N, K, rows_per_gate, dtype, absent):
    g = torch.Generator(device=dev).manual_seed(M + N + K)
    x, scale = L.quant_rowwise(torch.randn(M, K, generator=g, device=dev))
    w, ws = L.quant_rowwise(torch.randn(N, K, generator=g, device=dev) * 0.02)
    x[::5] = 0                                       # rows of zeros, negative ones where the weight's scale is negative
    ws[::3] *= -1
    scale[1::16] = float("inf")
    gate = torch.randn(M // rows_per_gate, N, generator=g, device=dev).to(dtype)
    residual = torch.randn(M, N, generator=g, device=dev).to(dtype)
    residual[::2, ::7], gate[:, ::11] = -0.0, 0.0
    gate[:, 1::13] *= 1e-4                            # products below binary16's normal numbers, with a residual that keeps them
    residual[1::2, 1::13] = 0.0
    scale[2::4] *= 1e-2
    plain = L.linear_w8a8(x, scale, w, ws, None, dtype, L.EPI_TORCH)
    want, rows = plain, gate.repeat_interleave(rows_per_gate, 0)
    if absent != "gate":
        want = rows * want
    if absent != "residual":
        want = residual + want
    guard = torch.full((M + 64, N), 7.0, dtype=dtype, device=dev)
    out = guard[:M]
    out.copy_(residual)
    L.linear_w8a8(x, scale, w, ws, None, dtype, L.EPI_TORCH, addend=None if absent == "residual" else out,
                  gate=None if absent == "gate" else gate, out=out)
    whole = torch.int32 if dtype == torch.float32 else torch.int16
    nan = want.isnan()
    assert torch.equal(out.isnan(), nan)
    assert torch.equal(out.view(whole)[~nan], want.view(whole)[~nan])
    assert bool((guard[M:] == 7.0).all())


@pytest.mark.gpu
def test_rows_wider_than_the_pieces_offsets(L, dev):
    """Columns beyond 2^27, which only a product over no columns at all has: sixteen rows of them exceed 32 bits."""
    M, N = 17, 2**28 + 8
    g = torch.Generator(device=dev).manual_seed(3)
    a, w = (torch.empty(n, 0, dtype=torch.int8, device=dev) for n in (M, N))
    draw = lambda *size: torch.empty(size, dtype=torch.bfloat16, device=dev).normal_(generator=g)
    bias, gate, residual = draw(N), draw(1, N), draw(M, N)
    call = lambda **kw: L.linear_w8a8(a, torch.ones(M, device=dev), w, 0.5, bias, torch.bfloat16, L.EPI_TORCH, addend=residual, gate=gate, **kw)
    want = [r + gate[0] * bias for r in residual]
    out = call()
    assert all(torch.equal(o, v) for o, v in zip(out, want))
    out.zero_()
    L.linear_w8a8_grouped([(a, torch.ones(M, device=dev), w, 0.5, bias, residual, gate)] * 2, torch.bfloat16, L.EPI_TORCH, outs=[out, out])
    assert all(torch.equal(o, v) for o, v in zip(out, want))
