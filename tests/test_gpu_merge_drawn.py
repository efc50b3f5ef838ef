"""The LoRA merge that draws its noise itself, against the merge on torch's own noise: the same bits."""
import ctypes

import pytest
import torch

# Shapes: elements below, at and beyond the generator's 524288 threads and its calls of four times as many (a partial last
# block, quarters that end inside a row); widths of one piece, of an odd number of 16, of several 256-column blocks and a rest;
# rows that fill no block of 32; every kind of rank (padded, four-wave, eight-wave workgroups).
CASES = [
    # N, K, rank, seed, scale per row, std of the factors
    (1, 16, 4, 27, True, 0.01), (17, 48, 12, -5, True, 0.01), (128, 4096, 16, 2**63 + 12345, True, 0.01), (513, 1040, 8, 1, False, 0.01),
    (2049, 1024, 32, 2, True, 0.01), (682, 3088, 20, 3, True, 0.01), (7, 524288, 4, 4, True, 0.01), (700, 12288, 64, 5, True, 0.01),
    (1000, 3072, 112, 6, True, 0.01), (333, 1552, 256, 7, True, 0.01), (4099, 2064, 48, 8, True, 0.01),
    (400, 2064, 8, 9, True, 10.0),       # every quotient far outside int8
    (400, 2064, 8, 10, True, 1e-20),     # products in the denormal range
    (400, 2064, 16, 11, True, 0.25),     # quotients of some tens: many elements are redone
    # every number of 16-rank steps that is built, on rows and columns around a tile's 32 and 128
    (31, 128, 16, 12, True, 0.01), (32, 144, 32, 13, True, 0.01), (33, 112, 48, 14, True, 0.01), (64, 272, 64, 15, False, 0.01),
    (65, 256, 80, 16, True, 0.01), (95, 368, 96, 17, True, 0.02), (97, 384, 112, 18, True, 0.02), (130, 400, 128, 19, True, 0.02),
    (161, 496, 160, 20, False, 0.02), (200, 528, 192, 21, True, 0.02), (223, 640, 224, 22, True, 0.02), (300, 784, 256, 23, True, 0.05),
    (3000, 272, 32, 24, True, 0.1),      # quotients that have to be saturated before they are added
    (640, 272, 256, 25, True, 0.5),      # an error bound that leaves a good part of the elements to the definition
]


@pytest.mark.gpu
@pytest.mark.parametrize("scale", [0.0, 1e-30, 1e-36, float("nan"), float("inf"), -0.001])
def test_drawn_merge_of_rows_without_a_usual_scale(pkg, L, dev, scale):
    """Single rows, which go to the list of open elements, and whole blocks of them, which are passed over and redone."""
    if not L.DRAWS_LIKE_TORCH:
        pytest.skip("this torch's generator is not the one that is reproduced")
    N, K, rank = 200, 400, 12
    g = torch.Generator(device=dev).manual_seed(5)
    w = torch.randint(-128, 128, (N, K), generator=g, device=dev, dtype=torch.int8)
    ws = torch.rand(N, generator=g, device=dev) * 0.002 + 0.0005
    ws[5] = scale
    ws[64:160] = scale
    up, down = torch.randn(N, rank, generator=g, device=dev) * 0.02, torch.randn(rank, K, generator=g, device=dev) * 0.02
    noise = pkg.int8_quant._draw_noise((N, K), 9, dev)
    drawn = L.lora_merge_sr_drawn(w, ws, pkg.int8_quant._seeded(9, dev), [(up, down, 1.0)], 0.75)
    assert torch.equal(drawn, L.lora_merge_sr(w, ws, noise, up=up, down=down, lora_scale=0.75))


@pytest.mark.gpu
@pytest.mark.parametrize("N,K,rank,seed,row,std", CASES)
def test_drawn_merge_equals_the_merge_on_torchs_noise(pkg, L, dev, N, K, rank, seed, row, std):
    if not L.DRAWS_LIKE_TORCH:
        pytest.skip("this torch's generator is not the one that is reproduced")
    g = torch.Generator(device=dev).manual_seed(N + K + rank)
    w = torch.randint(-128, 128, (N, K), generator=g, device=dev, dtype=torch.int8)
    ws = torch.rand(N if row else 1, generator=g, device=dev) * 0.002 + 0.0005
    up, down = torch.randn(N, rank, generator=g, device=dev) * std, torch.randn(rank, K, generator=g, device=dev) * std
    if N > 100:   # rows that have no quotient or leave the range of the approximate one
        up[3], up[5], up[6] = float("nan"), float("inf"), 0.0
        if row:
            ws[7], ws[8] = 1e-39, 3e7
    noise = pkg.int8_quant._draw_noise((N, K), seed, dev)
    drawn = L.lora_merge_sr_drawn(w, ws, pkg.int8_quant._seeded(seed, dev), [(up, down, 1.0)], 0.75)
    assert torch.equal(drawn, L.lora_merge_sr(w, ws, noise, up=up, down=down, lora_scale=0.75))


@pytest.mark.gpu
def test_drawn_merge_in_place(pkg, L, dev):
    if not L.DRAWS_LIKE_TORCH:
        pytest.skip("this torch's generator is not the one that is reproduced")
    N, K, rank = 301, 1040, 16
    w = torch.randint(-128, 128, (N, K), dtype=torch.int8, device=dev)
    up, down = torch.randn(N, rank, device=dev) * 0.05, torch.randn(rank, K, device=dev) * 0.05
    seeded = lambda: pkg.int8_quant._seeded(12, dev)
    want = L.lora_merge_sr_drawn(w, 0.003, seeded(), [(up, down, 1.0)])
    with pytest.MonkeyPatch.context() as m:
        m.setattr(torch, "empty_like", lambda t: t)   # (the result is written over the weight)
        got = L.lora_merge_sr_drawn(w, 0.003, seeded(), [(up, down, 1.0)])
    assert got is w and torch.equal(w, want)


@pytest.mark.gpu
def test_adapters_draw_what_they_drew(pkg, L, dev, monkeypatch):
    N, K = 640, 1040
    w = torch.randint(-127, 128, (N, K), dtype=torch.int8, device=dev)
    ws = torch.rand(N, 1, device=dev) * 0.002 + 0.0005
    lora = lambda r: (torch.randn(N, r, device=dev) * 0.02, torch.randn(r, K, device=dev) * 0.02, float(r), None, None, None)
    one = pkg.INT8LoRAPatchAdapter(set(), lora(16), ws, seed=7)
    stack = pkg.INT8MergedLoRAPatchAdapter([(pkg.INT8LoRAPatchAdapter(set(), lora(r), ws), 0.5) for r in (3, 9, 8)], ws, seed=8)
    full = pkg.INT8MergedLoRAPatchAdapter([(pkg.INT8LoRAPatchAdapter(set(), lora(r), ws), 1.3) for r in (1, 2, 1, 40, 12, 64, 128, 8)], ws, seed=9)
    nine = pkg.INT8MergedLoRAPatchAdapter([(pkg.INT8LoRAPatchAdapter(set(), lora(4), ws), 0.1 * i) for i in range(9)], ws, seed=10)
    empty = pkg.INT8MergedLoRAPatchAdapter([(pkg.INT8LoRAPatchAdapter(set(), lora(4), ws), 0.7),
                                            (pkg.INT8LoRAPatchAdapter(set(), (*lora(0)[:2], None, None, None, None), ws), 0.7)], ws, seed=11)
    adapters = (one, stack, full, nine, empty)
    drawn, taken = L.lora_merge_sr_drawn, []

    def watched(*a):
        merged = drawn(*a)
        taken.append(merged is not None)
        return merged

    monkeypatch.setattr(L, "lora_merge_sr_drawn", watched)
    now = [a.calculate_weight(w, "", 1.0, 1.0, None, None) for a in adapters]
    if L.DRAWS_LIKE_TORCH:   # nine LoRAs are too many for the launch: put side by side by torch, they are one
        assert taken == [True, True, True, False, True, True]
    monkeypatch.setattr(L, "DRAWS_LIKE_TORCH", False)
    for got, a in zip(now, adapters):
        assert torch.equal(got, a.calculate_weight(w, "", 1.0, 1.0, None, None))


@pytest.mark.gpu
def test_a_lora_of_strength_0_keeps_the_weight_and_the_fast_path(pkg, L, dev):
    if not L.DRAWS_LIKE_TORCH:
        pytest.skip("this torch's generator is not the one that is reproduced")
    N, K, rank = 12288, 3072, 32
    w = torch.randint(-128, 128, (N, K), dtype=torch.int8, device=dev)
    up, down = torch.randn(N, rank, device=dev) * 0.01, torch.randn(rank, K, device=dev) * 0.01
    generator = pkg.int8_quant._seeded(6, dev)
    merge = lambda lora_scale: L.lora_merge_sr_drawn(w, 0.002, generator, [(up, down, 1.0)], lora_scale)
    assert torch.equal(merge(0.0), w) and torch.equal(merge(-0.0), w)

    def median_time(lora_scale):
        times = []
        for _ in range(15):
            first, last = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            first.record()
            merge(lora_scale)
            last.record()
            torch.cuda.synchronize()
            times.append(first.elapsed_time(last))
        return sorted(times)[7]

    assert median_time(0.0) < 1.4 * median_time(1.0)   # (2.0 times where every element goes by the definition)
    up[5, 3], down[2, 7] = float("inf"), float("nan")   # sums that are not finite stay so at strength 0
    noise = pkg.int8_quant._draw_noise((N, K), 6, dev)
    assert torch.equal(merge(0.0), L.lora_merge_sr(w, 0.002, noise, up=up, down=down, lora_scale=0.0))


@pytest.mark.gpu
def test_rows_too_long_for_the_drawn_merge_are_merged_on_torchs_noise(pkg, L, dev):
    N, K, rank = 2, 1 << 24, 4
    w = torch.randint(-127, 128, (N, K), dtype=torch.int8, device=dev)
    up, down = torch.randn(N, rank, device=dev), torch.randn(rank, K, device=dev) * 0.01
    assert L.lora_merge_sr_drawn(w, 0.004, pkg.int8_quant._seeded(5, dev), [(up, down, 1.0)]) is None
    merged = pkg.INT8LoRAPatchAdapter(set(), (up, down, None, None, None, None), 0.004, seed=5).calculate_weight(w, "", 1.0, 1.0, None, None)
    assert torch.equal(merged, L.lora_merge_sr(w, 0.004, pkg.int8_quant._draw_noise((N, K), 5, dev), up=up, down=down))


@pytest.mark.gpu
def test_what_the_entry_point_refuses_is_left_to_the_caller(pkg, L, dev, monkeypatch):
    w = torch.randint(-127, 128, (32, 64), dtype=torch.int8, device=dev)
    up, down = torch.randn(32, 4, device=dev), torch.randn(4, 64, device=dev)
    assert L.lora_merge_sr_drawn(w, 0.004, pkg.int8_quant._seeded(5, dev), [(up, down, 1.0)]) is not None
    monkeypatch.setattr(L.lib(), "i8f_lora_merge_sr_drawn", lambda *a: L.ERR_UNSUPPORTED)
    assert L.lora_merge_sr_drawn(w, 0.004, pkg.int8_quant._seeded(5, dev), [(up, down, 1.0)]) is None


def test_drawn_merge_refuses_what_it_cannot_do(L):
    one, null = ctypes.c_void_p(4096), None
    INVALID, UNSUPPORTED = -1, -2

    def call(w=one, factors=((4096, 4096, 8),), lanes=256, N=4, K=16, ws=one, mode=0, nbytes=None):
        arr = (L._LoraFactors * max(1, len(factors)))(*((u, d, r, 1.0) for u, d, r in factors))
        size = L.lib().i8f_lora_merge_sr_drawn_workspace_bytes(N, K, sum(r for _, _, r in factors), len(factors))
        return L.lib().i8f_lora_merge_sr_drawn(w, ws, 1.0, mode, arr, len(factors), 1.0, 0, lanes, N, K, one, one,
                                               size if nbytes is None else nbytes, null)

    assert call(w=null) == INVALID and call(factors=((None, 4096, 8),)) == INVALID and call(factors=()) == INVALID and call(lanes=0) == INVALID
    assert call(factors=((4096, 4096, 0),)) == INVALID and call(ws=null, mode=1) == INVALID and call(mode=2) == INVALID
    assert call(nbytes=127) == INVALID and call(N=-1) == INVALID
    assert call(factors=((4096, 4096, 4), (4096, 4096, 4)), nbytes=256) == INVALID          # the factors side by side need room
    assert call(K=24) == UNSUPPORTED and call(factors=((4096, 4096, 6),)) == UNSUPPORTED and call(lanes=100) == UNSUPPORTED
    assert call(factors=((4096, 4096, 260),)) == UNSUPPORTED and call(factors=((4096, 4096, 129), (4096, 4096, 128))) == UNSUPPORTED
    assert call(factors=((4096, 4096, 4),) * 9) == UNSUPPORTED and call(factors=((4100, 4096, 8),)) == UNSUPPORTED
    assert call(N=2**25 + 1) == UNSUPPORTED and call(N=1, K=2**24) == UNSUPPORTED and call(lanes=2**24 + 256) == UNSUPPORTED
    assert call(N=2**24) == UNSUPPORTED      # more calls of the generator than a launch has blocks
    assert call(N=0) == 0 and call(K=0) == 0


def force(L, monkeypatch, form):
    """From here on the drawn merge takes form 0 (few elements) or 1."""
    lib = L.lib()
    run, size = lib.i8f_internal_merge_drawn, lib.i8f_internal_merge_drawn_workspace_bytes
    run.argtypes = [ctypes.c_int, *lib.i8f_lora_merge_sr_drawn.argtypes]
    size.argtypes, size.restype = [ctypes.c_int, *lib.i8f_lora_merge_sr_drawn_workspace_bytes.argtypes], ctypes.c_int64
    monkeypatch.setattr(lib, "i8f_lora_merge_sr_drawn", lambda *a: run(form, *a))
    monkeypatch.setattr(lib, "i8f_lora_merge_sr_drawn_workspace_bytes", lambda *a: size(form, *a))


@pytest.mark.gpu
@pytest.mark.parametrize("N,K,rank,seed,row,std", CASES)
@pytest.mark.parametrize("form", [0, 1])
def test_both_forms_of_the_drawn_merge(pkg, L, dev, monkeypatch, form, N, K, rank, seed, row, std):
    force(L, monkeypatch, form)
    if form == 0 and rank > 224:
        assert L.lora_merge_sr_drawn(torch.zeros(N, K, dtype=torch.int8, device=dev), 0.5, pkg.int8_quant._seeded(seed, dev),
                                     [(torch.zeros(N, rank, device=dev), torch.zeros(rank, K, device=dev), 1.0)]) is None
    else:
        test_drawn_merge_equals_the_merge_on_torchs_noise(pkg, L, dev, N, K, rank, seed, row, std)


@pytest.mark.gpu
@pytest.mark.parametrize("form", [0, 1])
@pytest.mark.parametrize("scale", [0.0, 1e-30, float("nan"), -0.001])
def test_both_forms_of_rows_without_a_usual_scale(pkg, L, dev, monkeypatch, form, scale):
    force(L, monkeypatch, form)
    test_drawn_merge_of_rows_without_a_usual_scale(pkg, L, dev, scale)


@pytest.mark.gpu
@pytest.mark.parametrize("form", [0, 1])
@pytest.mark.parametrize("N,K,ranks", [(33, 48, (3, 9, 8)), (640, 1040, (16, 32, 64)), (1025, 2064, (4, 4)), (40, 272, (1, 2, 1, 40, 12, 64, 72, 8))])
def test_both_forms_of_a_stack(pkg, L, dev, monkeypatch, form, N, K, ranks):
    if not L.DRAWS_LIKE_TORCH:
        pytest.skip("this torch's generator is not the one that is reproduced")
    force(L, monkeypatch, form)
    g = torch.Generator(device=dev).manual_seed(N)
    w = torch.randint(-128, 128, (N, K), generator=g, device=dev, dtype=torch.int8)
    parts = [(torch.randn(N, r, generator=g, device=dev) * 0.02, torch.randn(r, K, generator=g, device=dev) * 0.02, 0.3 * i - 0.5) for i, r in enumerate(ranks)]
    got = L.lora_merge_sr_drawn(w, 0.002, pkg.int8_quant._seeded(3, dev), parts)
    up, down = torch.cat([u for u, _, _ in parts], 1), torch.cat([d * m for _, d, m in parts])
    assert torch.equal(got, L.lora_merge_sr(w, 0.002, pkg.int8_quant._draw_noise((N, K), 3, dev), up=up, down=down))


def test_which_form_the_drawn_merge_takes(L):
    """By the memory that it asks for: the form for few elements has two bytes of noise to an element."""
    size = L.lib().i8f_lora_merge_sr_drawn_workspace_bytes
    up256 = lambda n: -(-n // 256) * 256
    few = lambda N, K, rank, count=1: size(N, K, rank, count) == up256(2 * N * K) + (up256(4 * N * rank) + 4 * K * rank if count > 1 else 0)
    assert few(16, 3072, 16) and few(1024, 1024, 16) and few(1024, 1024, 64) and few(3072, 3072, 8) and few(2048, 1024, 32)
    assert few(3840, 3840, 8) and few(12288, 3072, 8) and few(18432, 3072, 4) and few(1280, 1280, 32, 2) and few(944, 768, 16)
    assert not few(1024, 1024, 256) and not few(2048, 2048, 128) and not few(3072, 3072, 64) and not few(12288, 12288, 4)
    assert not few(12288, 3072, 32) and not few(9216, 3072, 112, 3) and not few(1168, 1632, 72, 3) and not few(392, 10016, 68, 2)


@pytest.mark.gpu
@pytest.mark.parametrize("N,K,rank", [(640, 18432, 16), (333, 18448, 28), (1000, 11008, 8), (5, 20480, 4)])
def test_two_workgroups_to_a_cu(pkg, L, dev, monkeypatch, N, K, rank):
    """Widths whose panels leave a good part of the CUs without one, full and with a rest (5 rows: not enough for it)."""
    force(L, monkeypatch, 1)
    test_drawn_merge_equals_the_merge_on_torchs_noise(pkg, L, dev, N, K, rank, 4, True, 0.01)


@pytest.mark.gpu
@pytest.mark.parametrize("form", [0, 1])
def test_both_forms_in_place(pkg, L, dev, monkeypatch, form):
    force(L, monkeypatch, form)
    test_drawn_merge_in_place(pkg, L, dev)


@pytest.mark.gpu
def test_a_generator_of_few_threads_takes_a_launch_for_the_factors_of_its_own(L, dev):
    """256 threads: the calls of the generator and the blocks for a stack's factors are more rows of blocks than a launch has."""
    N, K, ranks, lib = 4096, 16368, (4, 4), L.lib()
    run, size = lib.i8f_internal_merge_drawn, lib.i8f_internal_merge_drawn_workspace_bytes
    run.argtypes = [ctypes.c_int, *lib.i8f_lora_merge_sr_drawn.argtypes]
    size.argtypes, size.restype = [ctypes.c_int, *lib.i8f_lora_merge_sr_drawn_workspace_bytes.argtypes], ctypes.c_int64
    g = torch.Generator(device=dev).manual_seed(8)
    w = torch.randint(-128, 128, (N, K), generator=g, device=dev, dtype=torch.int8)
    parts = [(torch.randn(N, r, generator=g, device=dev) * 0.02, torch.randn(r, K, generator=g, device=dev) * 0.02) for r in ranks]
    arr = (L._LoraFactors * 2)(*((u.data_ptr(), d.data_ptr(), u.shape[1], 0.5) for u, d in parts))
    outs = []
    for form in (0, 1):
        out, scratch = torch.empty_like(w), torch.empty(size(form, N, K, sum(ranks), 2), dtype=torch.uint8, device=dev)
        assert run(form, w.data_ptr(), None, 0.002, L.SCALE_TENSOR, arr, 2, 1.0, 5, 256, N, K, out.data_ptr(), scratch.data_ptr(), scratch.numel(),
                   torch.cuda.current_stream().cuda_stream) == 0
        outs.append(out)
    assert torch.equal(*outs) and not torch.equal(outs[0], w)
