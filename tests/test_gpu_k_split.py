"""The K split below K = 10240 and its exchange with one to seven other slices: the bits of the call without a workspace."""
import pytest
import torch


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,dtype", [
    (128, 1536, 6144, torch.bfloat16), (17, 384, 6160, torch.float16), (64, 3072, 7168, torch.bfloat16), (33, 1024, 8192, torch.bfloat16),
    (512, 1024, 8192, torch.float16), (512, 3072, 9216, torch.bfloat16), (20, 400, 10224, torch.float32),                  # 2 to 4 slices
    (64, 3072, 12288, torch.bfloat16), (17, 512, 12288, torch.bfloat16), (40, 512, 14336, torch.float16), (17, 520, 16384, torch.bfloat16),  # 5 to 8
])
def test_split_gives_the_bits_of_the_unsplit_product(L, dev, M, N, K, dtype):
    g = torch.Generator(device=dev).manual_seed(M + N + K)
    x, s = L.quant_rowwise(torch.randn(M, K, generator=g, device=dev).bfloat16())
    w, ws = L.quant_rowwise(torch.randn(N, K, generator=g, device=dev) * 0.02)
    gate, residual = torch.randn(1, N, generator=g, device=dev).to(dtype), torch.randn(M, N, generator=g, device=dev).to(dtype)
    plain = torch.empty(M, N, device=dev, dtype=dtype)
    ws = ws.reshape(-1)
    assert L.lib().i8f_linear_w8a8(x.data_ptr(), s.data_ptr(), w.data_ptr(), ws.data_ptr(), 0.0, L.SCALE_ROW, None, L.BF16, plain.data_ptr(),
                                   L.dtype_code(dtype), M, N, K, L.EPI_TORCH, torch.cuda.current_stream().cuda_stream) == 0
    for _ in range(3):
        assert torch.equal(L.linear_w8a8(x, s, w, ws, None, dtype, L.EPI_TORCH), plain)
    assert torch.equal(L.linear_w8a8(x, s, w, ws, None, dtype, L.EPI_TORCH, addend=residual, gate=gate), residual + gate * plain)
    work = L._splitk_workspace(x, M, N, K)
    assert work is not None and int(work[:4096].view(torch.int32).abs().sum()) == 0


@pytest.mark.gpu
@pytest.mark.parametrize("K", [8192, 10240])
def test_split_inside_a_graph(L, dev, K):
    M, N = 33, 1024
    x, s = L.quant_rowwise(torch.randn(M, K, device=dev).bfloat16())
    w, ws = L.quant_rowwise(torch.randn(N, K, device=dev) * 0.02)
    want = L.linear_w8a8(x, s, w, ws, None, torch.bfloat16, L.EPI_TORCH)
    out = torch.empty_like(want)
    graph = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph):
        L.linear_w8a8(x, s, w, ws, None, torch.bfloat16, L.EPI_TORCH, out=out)
    for _ in range(4):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want)
        assert torch.equal(L.linear_w8a8(x, s, w, ws, None, torch.bfloat16, L.EPI_TORCH), want)
