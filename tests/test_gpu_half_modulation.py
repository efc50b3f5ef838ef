"""The packed binary16 modulation in the quantiser, against torch's own operations on a whole grid of magnitudes.
(Separate operations: the fused spelling is not packed; it rounds its sum to binary32 first, which shows against addcmul
where a shift of 2^-24 decides a tie.)"""
import pytest
import torch


@pytest.mark.gpu
@pytest.mark.parametrize("rotate", [False, True])
@pytest.mark.parametrize("M,K", [(3, 128), (5, 3840), (1030, 1152)])   # one group of lanes, a partial last run, many workgroups
def test_half_modulation_equals_torchs_operations(L, dev, M, K, rotate):
    g = torch.Generator(device=dev).manual_seed(M + K)
    # every exponent from the denormals to the largest, both signs; products and sums that overflow, vanish and cancel
    def spread(*shape):
        e = torch.randint(-24, 16, shape, generator=g, device=dev).float()
        return ((torch.rand(*shape, generator=g, device=dev) + 1.0) * torch.exp2(e) * torch.randn(*shape, generator=g, device=dev).sign()).half()
    x, s, t = spread(M, K), spread(1, K), spread(1, K)
    if rotate:   # (a sum of 128 values of which one is infinite tells nothing)
        x, s, t = x.clamp(-8, 8), s.clamp(-8, 8), t.clamp(-8, 8)
    s[0, :8] = -1.0          # a gain of zero
    q, scale = L.quant_rowwise(x, rotate=rotate, prologue=L.PRO_MODULATE, mod_scale=s, mod_shift=t)
    y = (1 + s) * x + t
    want_q, want_scale = L.quant_rowwise(y, rotate=rotate)
    assert torch.equal(q, want_q) and torch.equal(scale.view(torch.int32), want_scale.view(torch.int32))
