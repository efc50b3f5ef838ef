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


UNTOUCHED = 0x5a5a5a5a   # (no sum of 16384 products)


def partials(L, work):
    return work[L._SPLITK_COUNTER_BYTES:].view(torch.int32)


def words_of(M, N, tile, slices):
    return 0 if slices == 1 else slices * (-(-M // tile[0]) * tile[0]) * (-(-N // tile[1]) * tile[1])


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,tile,slices", [
    (128, 1536, 6144, (64, 64), 3), (17, 384, 6160, (64, 64), 3), (64, 3072, 7168, (64, 64), 3), (512, 1024, 8192, (64, 64), 2),
    (512, 3072, 9216, (128, 96), 2), (20, 400, 10224, (64, 64), 4), (1024, 2048, 12288, (128, 128), 2), (256, 3072, 12288, (128, 96), 4),
    (64, 3072, 12288, (64, 64), 5), (17, 512, 12288, (64, 64), 6), (40, 512, 14336, (64, 64), 7), (17, 520, 16384, (64, 64), 8),
    (17, 384, 6128, (64, 64), 1), (512, 1024, 6128, (64, 64), 1), (256, 3072, 9216, (64, 64), 1), (512, 2048, 6144, (64, 64), 1),
    (1000, 1000, 6144, (64, 64), 1),
])
def test_how_many_slices_a_shape_takes(L, dev, M, N, K, tile, slices):
    """By the partial sums that the launch leaves in the workspace: every slice of every tile writes its own."""
    g = torch.Generator(device=dev).manual_seed(M + N + K)
    x, s = L.quant_rowwise(torch.randn(M, K, generator=g, device=dev).bfloat16())
    w, ws = L.quant_rowwise(torch.randn(N, K, generator=g, device=dev) * 0.02)
    ws, out = ws.reshape(-1), torch.empty(M, N, device=dev, dtype=torch.bfloat16)
    work = torch.zeros(L.lib().i8f_linear_w8a8_workspace_bytes(), dtype=torch.uint8, device=dev)
    partials(L, work).fill_(UNTOUCHED)
    assert L.lib().i8f_linear_w8a8_splitk(x.data_ptr(), s.data_ptr(), w.data_ptr(), ws.data_ptr(), 0.0, L.SCALE_ROW, None, L.BF16, None, out.data_ptr(),
                                          L.BF16, M, N, K, L.EPI_TORCH, work.data_ptr(), work.numel(), torch.cuda.current_stream().cuda_stream) == 0
    assert torch.equal(out, L.linear_w8a8(x, s, w, ws, None, torch.bfloat16, L.EPI_TORCH))
    assert int((partials(L, work) != UNTOUCHED).sum()) == words_of(M, N, tile, slices)


@pytest.mark.gpu
@pytest.mark.parametrize("K,slices", [(8192, 1), (10224, 1), (10240, 5)])
def test_below_10240_a_captured_call_is_not_split(L, dev, monkeypatch, K, slices):
    M, N = 33, 1024
    x, s = L.quant_rowwise(torch.randn(M, K, device=dev).bfloat16())
    w, ws = L.quant_rowwise(torch.randn(N, K, device=dev) * 0.02)
    want = L.linear_w8a8(x, s, w, ws, None, torch.bfloat16, L.EPI_TORCH)
    handed, ask = [], L._splitk_workspace
    monkeypatch.setattr(L, "_splitk_workspace", lambda *a: handed.append(ask(*a)) or handed[-1])
    graph = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph):
        out = L.linear_w8a8(x, s, w, ws, None, torch.bfloat16, L.EPI_TORCH)
    assert (handed[0] is not None) == (slices > 1)
    for _ in range(3):
        out.zero_()
        if slices > 1:
            partials(L, handed[0]).fill_(UNTOUCHED)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want)
        assert slices == 1 or int((partials(L, handed[0]) != UNTOUCHED).sum()) == words_of(M, N, (64, 64), slices)
