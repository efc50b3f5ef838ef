"""The W8A16 layer of up to 16 rows with one, two and three 16-column blocks to a workgroup: a column's sum does not depend on the
form, so a layer equals, bit for bit, its columns taken 4096 at a time (one block to a workgroup, which the oracle's tests cover)."""
import pytest
import torch

# either side of 256, 512 and 768 blocks, last workgroups with one column block or a part of one; K of whole steps and not
SHAPES = [(1, 4104, 2560), (7, 4104, 144), (16, 8192, 272), (6, 8192, 2576), (1, 8200, 2304), (9, 8216, 144), (3, 10000, 3072),
          (16, 12280, 400), (1, 12288, 2304), (8, 12288, 2288), (2, 12304, 3072)]


def _layer(L, dev, M, N, K, dtype):
    g = torch.Generator(device=dev).manual_seed(M + N + K)
    x = torch.randn(M, K, generator=g, device=dev).to(dtype)
    w = torch.randint(-128, 128, (N, K), generator=g, device=dev, dtype=torch.int8)
    return x, w, torch.rand(N, 1, generator=g, device=dev) * 0.02, torch.randn(N, generator=g, device=dev).to(dtype)


def _in_pieces(L, x, w, ws, b):
    cuts = [(n, min(n + 4096, w.shape[0])) for n in range(0, w.shape[0], 4096)]
    return torch.cat([L.linear_w8a16_small_m(x, w[i:j], ws[i:j], b[i:j]) for i, j in cuts], 1)


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", SHAPES)
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_columns_do_not_depend_on_how_many_share_a_workgroup(L, dev, M, N, K, dtype):
    x, w, ws, b = _layer(L, dev, M, N, K, dtype)
    assert torch.equal(L.linear_w8a16_small_m(x, w, ws, b), _in_pieces(L, x, w, ws, b))


@pytest.mark.gpu
@pytest.mark.parametrize("M,Ns,K", [(1, (4096, 16), 2560), (7, (4104, 4088), 144), (1, (6152, 2048), 2304), (16, (40, 8200, 2000), 144),
                                    (1, (4096, 4096, 4096), 2304), (2, (4097, 3, 4000, 4188), 2560)])
def test_layers_in_one_launch_take_the_same_forms(L, dev, M, Ns, K):
    layers = [_layer(L, dev, M, N, K, torch.bfloat16) for N in Ns]
    for layer, got in zip(layers, L.linear_w8a16_small_m_grouped(layers)):
        assert torch.equal(got, _in_pieces(L, *layer))
