"""Each kernel alone against a plain float64 formula, at sizes other than the engine's."""
import math

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


def rnd(*shape, seed=0, scale=1.0, dtype=torch.float32):
    g = torch.Generator().manual_seed(seed)
    return (torch.randn(*shape, generator=g, dtype=torch.float64) * scale).to(dtype)


def to_dev(t, dtype=None):
    return t.to(device=DEV, dtype=dtype or t.dtype).contiguous()


# ----------------------------------------------------------------------- products
# (rows of W, k, tokens): the awkward shapes of the reference's own matmul test
# (crates/glassbox-core/src/kernels.rs:697) and larger ones that cross tile edges
GEMM_SHAPES_F32 = [(1, 32, 1), (8, 64, 2), (17, 64, 3), (33, 96, 9), (50, 160, 17), (331, 100, 70), (130, 257, 129),
                   # few rows through the skinny kernel: a k of one slice and a part, of many groups of slices, rows of W
                   # that do not fill the last workgroup, rows of A in several passes
                   (2048, 2048, 1), (50, 100, 5), (2048, 8192, 8), (331, 2120, 16), (96, 4100, 33), (1000, 72, 64),
                   (130, 258, 7)]
GEMM_SHAPES_BF16 = [(1, 32, 1), (8, 64, 2), (17, 64, 3), (33, 96, 9), (50, 160, 17), (331, 104, 64), (331, 104, 65),
                    (130, 264, 129), (16, 2048, 8), (272, 72, 300), (49, 520, 33),
                    # few rows of W and a long k: the skinny kernels split k over the waves of a workgroup
                    (2048, 2048, 8), (2048, 8192, 8), (64, 2056, 1), (100, 4104, 33), (2048, 2048, 64), (48, 8192, 17),
                    # the tiled kernel over many k-steps, k a multiple of its step and not, one and two
                    # k-steps of prefetch (few and many tiles), fewer k-steps than the prefetch reaches
                    (512, 1024, 200), (2048, 2048, 130), (96, 8192, 70), (1536, 1088, 520), (200, 128, 66), (3000, 192, 300),
                    (640, 1032, 257),
                    # a k of twelve to fifteen 64-wide blocks on sixteen waves (some of which find no block, or a part of one)
                    (960, 960, 12), (2560, 960, 33), (1600, 776, 20), (5120, 1016, 64)]


@pytest.mark.parametrize("N,K,M", GEMM_SHAPES_F32)
@pytest.mark.parametrize("accumulate", [False, True])
def test_gemm_f32(N, K, M, accumulate):
    from glassbox_amd import ops
    a, w, c0 = rnd(M, K, seed=1), rnd(N, K, seed=2), rnd(M, N, seed=3)
    want = a.double() @ w.double().T + (c0.double() if accumulate else 0)
    c = to_dev(c0.clone())
    ops.gemm(to_dev(a), to_dev(w), c, accumulate=accumulate)
    err = (c.cpu().double() - want).abs().max().item()
    assert err <= 1e-4 * (1 + want.abs().max().item()), err   # kernels.rs:716 tolerance


@pytest.mark.parametrize("N,K", [(1, 32), (50, 160), (17, 64), (331, 100), (96, 4100), (2048, 2048), (512, 8192), (8, 16384)])
def test_gemm_f32_is_summed_in_one_order_by_both_kernels_and_at_every_number_of_rows(N, K):
    """A cell's sum is cut into slices of 64 of k, each a chain of fused multiply-adds from zero, added in order
    (``csrc/hip/gemm_f32.hip``): the skinny kernel (4, 8 or 16 rows of W a workgroup, a lane a slice) and the tiled one give the
    same bits, and a row of A gives the same bits alone, among 8 and among 70 rows, which is what lets batched
    and unbatched generation agree exactly in 32-bit."""
    from glassbox_amd import ops
    lib = ops._lib("gemm_f32")
    stream = torch.cuda.current_stream().cuda_stream
    a, w = to_dev(rnd(70, K, seed=5)), to_dev(rnd(N, K, seed=6))
    c0 = to_dev(rnd(70, N, seed=7))

    def run(rows, which, accumulate):
        c = c0[:rows].clone()
        rc = lib.gb_gemm_f32_by(a.data_ptr(), K, w.data_ptr(), K, c.data_ptr(), N, rows, N, K, accumulate, which, stream)
        assert rc == 0, lib.gb_last_error().decode()
        return c.cpu()

    for accumulate in (0, 1):
        tiled = run(70, 1, accumulate)
        want = a.cpu().double() @ w.cpu().double().T + (c0.cpu().double() if accumulate else 0)
        assert (tiled.double() - want).abs().max().item() <= 1e-4 * (1 + want.abs().max().item())
        for rows in (1, 2, 3, 8, 13, 16, 17, 40, 64):
            skinny = run(rows, 2, accumulate)
            assert torch.equal(skinny, tiled[:rows]), f"{rows} rows: the skinny kernel's bits differ from the tiled kernel's"
            assert torch.equal(run(rows, 1, accumulate), tiled[:rows]), f"{rows} rows: the tiled kernel's bits depend on M"
    # the skinny kernel is refused where it does not apply, not run wrongly
    assert lib.gb_gemm_f32_by(a.data_ptr(), K, w.data_ptr(), K, c0.data_ptr(), N, 70, N, K, 0, 2, stream) == 1
    assert "skinny" in lib.gb_last_error().decode()


@pytest.mark.parametrize("N,K,M", [(331, 100, 200), (130, 260, 129), (2048, 2048, 300), (512, 8192, 65), (96, 4100, 331),
                                   (257, 16, 128), (128, 72, 1)])
def test_gemm_f32_wide_kernel_gives_the_bits_of_the_tiled_kernel(N, K, M):
    """The kernel for prompts (128 x 128 of C a workgroup on the matrix cores, two k-steps in LDS) keeps the one
    summation order: the same bits as the tiled kernel, with and without accumulation, on tiles that hang over
    every edge; and it is refused where rows are no 16-byte words."""
    from glassbox_amd import ops
    lib = ops._lib("gemm_f32")
    stream = torch.cuda.current_stream().cuda_stream
    a, w, c0 = to_dev(rnd(M, K, seed=11)), to_dev(rnd(N, K, seed=12)), to_dev(rnd(M, N, seed=13))
    for accumulate in (0, 1):
        got = {}
        for which in (1, 3):
            c = c0.clone()
            rc = lib.gb_gemm_f32_by(a.data_ptr(), K, w.data_ptr(), K, c.data_ptr(), N, M, N, K, accumulate, which, stream)
            assert rc == 0, lib.gb_last_error().decode()
            got[which] = c.cpu()
        want = a.cpu().double() @ w.cpu().double().T + (c0.cpu().double() if accumulate else 0)
        assert (got[1].double() - want).abs().max().item() <= 1e-4 * (1 + want.abs().max().item())
        assert torch.equal(got[3], got[1]), "the wide kernel's bits differ from the tiled kernel's"
    if K > 4:
        assert lib.gb_gemm_f32_by(a.data_ptr() + 4, K, w.data_ptr(), K, c0.data_ptr(), N, M, N, K - 4, 0, 3, stream) == 1
        assert "wide" in lib.gb_last_error().decode()


@pytest.mark.parametrize("N,K,M", [(33, 64, 31), (32, 68, 33), (65, 260, 64), (31, 1024, 1), (960, 2564, 9), (8, 512, 200),
                                   # as dispatched: 8 and 16 rows of W a workgroup, and few rows by so many of W that the wide
                                   # kernel's tiles would do, on either side of where it begins
                                   (3077, 580, 1), (3077, 580, 2), (3077, 580, 4), (3077, 1284, 6), (4105, 260, 2), (24600, 68, 64),
                                   (24600, 68, 65)])
def test_gemm_f32_matrix_core_kernels_round_as_the_tiled_kernel_does(N, K, M):
    """The wide and the sliced kernel (four and eight waves; fewer slices than waves, one more, a last slice that k cuts) and
    the product as it is dispatched give the bits of the tiled kernel's chains of fmaf: products that are denormal, huge
    and cancelling ones, infinities and NaN in a row of each operand."""
    from glassbox_amd import ops
    lib = ops._lib("gemm_f32")
    stream = torch.cuda.current_stream().cuda_stream
    a, w, c0 = rnd(M, K, seed=21), rnd(N, K, seed=22), rnd(M, N, seed=23)
    a[0] *= 1e-22
    w[0] *= 1e-19
    a[M // 2, K - 1], w[N // 2, 0], w[N - 1, K // 2] = float("inf"), 3e38, float("nan")
    a, w, c0 = to_dev(a), to_dev(w), to_dev(c0)
    for accumulate in (0, 1):
        got = {}
        for which in (1, 0, 3, 4, 5):
            c = c0.clone()
            rc = lib.gb_gemm_f32_by(a.data_ptr(), K, w.data_ptr(), K, c.data_ptr(), N, M, N, K, accumulate, which, stream)
            assert rc == 0, lib.gb_last_error().decode()
            got[which] = c.cpu()
        assert torch.isnan(got[1]).any() and not torch.isnan(got[1]).all()
        for which in (0, 3, 4, 5):
            assert torch.equal(torch.isnan(got[which]), torch.isnan(got[1]))
            assert torch.equal(torch.nan_to_num(got[which], 0.25), torch.nan_to_num(got[1], 0.25)), which


@pytest.mark.parametrize("M,K,inter,nh,nkv,hd", [
    (1, 960, 2560, 15, 5, 64), (2, 576, 1536, 9, 3, 64),      # 16, 8 and 4 rows of W a workgroup
    (1, 2560, 23, 3, 0, 2), (2, 1280, 1025, 2, 1, 6),         # the longest rows that a workgroup norms; pairs that a workgroup shares
    (1, 4, 1, 1, 1, 20), (2, 252, 130, 5, 5, 100), (2, 260, 2049, 2, 1, 258), (1, 1028, 600, 33, 1, 64)])
def test_gemm_step_f32_gives_the_bits_of_the_kernels_it_replaces(M, K, inter, nh, nkv, hd):
    """Norm, product and gated unit, or norm, product, rotation and cache write, in one launch (csrc/hip/gemm_f32.hip,
    StepExtras): the bits of the four kernels one after the other, with and without the norm, the angles and the pages."""
    from glassbox_amd import ops
    x, gamma = to_dev(rnd(M, K, seed=31) * 3), to_dev(rnd(K, seed=32))
    wu, wh = to_dev(rnd(2 * inter, K, seed=33)), to_dev(rnd((nh + 2 * nkv) * hd, K, seed=34))
    f32 = lambda *shape: torch.zeros(shape, dtype=torch.float32, device=DEV)
    h = f32(M, K)
    ops.rmsnorm(x, gamma, 1e-5, h)
    pos = torch.tensor([5, 77][:M], dtype=torch.int32, device=DEV)
    cos, sin = f32(M, hd // 2), f32(M, hd // 2)
    ops.rope_table(pos, to_dev(rnd(hd // 2, seed=35).abs()), cos, sin)
    slots = torch.tensor([18, 3][:M], dtype=torch.int32, device=DEV)
    ran = 0
    for rms in (None, (gamma, 1e-5)):
        rows = h if rms else x
        if ops.step_f32_takes(M, 2 * inter, K, rms is not None):
            gu, want, got = f32(M, 2 * inter), f32(M, inter), f32(M, inter)
            ops.gemm(rows, wu, gu)
            ops.silu_mul(gu, want)
            ops.gemm_step_f32(x, wu, got, rms=rms, silu_mul=True)
            assert torch.equal(got, want)
            ran += 1
        if not ops.step_f32_takes(M, wh.shape[0], K, rms is not None):
            continue
        for angles in ((cos, sin), (None, None)):
            for store in (True, False):
                if store and nkv == 0:
                    continue
                outs = []
                for fused in (False, True):
                    qkv = f32(M, wh.shape[0])
                    kp = torch.zeros(ops.key_pages_shape(2, max(nkv, 1), 16, hd), device=DEV)
                    vp = f32(2, max(nkv, 1), hd, 16)
                    place = (slots, kp, vp) if store else (None, None, None)
                    if fused:
                        ops.gemm_step_f32(x, wh, qkv, rms=rms, heads=(nh, nkv, hd, *angles, *place))
                    else:
                        ops.gemm(rows, wh, qkv)
                        ops.rope_store(qkv, *angles, *place, nh, nkv, hd, rotate=angles[0] is not None)
                    outs.append((qkv, kp, vp))
                for got, want in zip(outs[1], outs[0]):
                    assert torch.equal(got, want)
                ran += 1
    assert ran
    # refused where it does not apply
    assert not ops.step_f32_takes(M, 2, 2564 if M == 1 else 1284, True) and not ops.step_f32_takes(3, 64, 64, False)
    # nor, with the norm, before very many rows of W of a short k
    assert not ops.step_f32_takes(M, 16384, 508, True) and ops.step_f32_takes(M, 16384, 512, True) and ops.step_f32_takes(M, 16384, 508, False)
    assert ops.step_f32_takes(M, 8192, 64, True) and not ops.step_f32_takes(M, 8194, 64, True)
    with pytest.raises(ops.KernelError):
        ops.gemm_step_f32(to_dev(rnd(3, 64)), to_dev(rnd(8, 64)), f32(3, 8))


def test_gemm_f32_takes_rows_that_are_no_words_of_16_bytes():
    """A k that is no multiple of 4, or operands that start in the middle of a word, go through the tiled kernel."""
    from glassbox_amd import ops
    for K, off in ((30, 0), (32, 1), (257, 0)):
        a, w = rnd(5, K + off, seed=8), rnd(20, K + off, seed=9)
        c = to_dev(torch.zeros(5, 20))
        da, dw = to_dev(a)[:, off:], to_dev(w)[:, off:]
        ops.gemm(da, dw, c)
        want = a[:, off:].double() @ w[:, off:].double().T
        assert (c.cpu().double() - want).abs().max().item() <= 1e-4 * (1 + want.abs().max().item())


@pytest.mark.parametrize("N,K,M", GEMM_SHAPES_BF16)
@pytest.mark.parametrize("out", ["bf16", "f32", "f32+"])
def test_gemm_bf16(N, K, M, out):
    from glassbox_amd import ops
    a, w = rnd(M, K, seed=1).bfloat16(), rnd(N, K, seed=2).bfloat16()
    c0 = rnd(M, N, seed=3)
    want = a.double() @ w.double().T + (c0.double() if out == "f32+" else 0)
    c = to_dev(c0.clone(), torch.bfloat16 if out == "bf16" else torch.float32)
    ops.gemm(to_dev(a), to_dev(w), c, accumulate=(out == "f32+"))
    got = c.cpu().double()
    # products of bfloat16 numbers are exact in 32-bit; only the summation order and (for a
    # bfloat16 result) the final rounding differ from the float64 sum
    tol = 1e-4 * math.sqrt(K) + (2 ** -8) * want.abs().max().item() * (out == "bf16")
    assert (got - want).abs().max().item() <= tol


@pytest.mark.parametrize("I,K,M", [(8, 32, 1), (176, 64, 5), (144, 80, 16), (200, 2048, 17), (8192, 2048, 8), (88, 4104, 64),
                                   # more than 64 rows: the tiled kernel's epilogue
                                   (176, 64, 130), (72, 264, 65), (1024, 520, 300), (2560, 960, 200), (2560, 960, 400), (1000, 2048, 129)])
def test_gemm_bf16_fused_silu_mul(I, K, M):
    """Stacked gate/up rows with the activation applied in the product's epilogue
    (crates/glassbox-core/src/model.rs:335-340), against the formula in float64."""
    from glassbox_amd import ops
    a, w = rnd(M, K, seed=1).bfloat16(), (rnd(2 * I, K, seed=2) / math.sqrt(K)).bfloat16()
    gu = a.double() @ w.double().T
    g, u = gu[:, :I], gu[:, I:]
    want = g / (1 + torch.exp(-g)) * u
    for dt in (torch.bfloat16, torch.float32):
        out = torch.full((M, I), 7.0, device=DEV, dtype=dt)
        ops.gemm(to_dev(a), to_dev(w), out, silu_mul=True)
        tol = 1e-4 + (2 ** -8) * want.abs().max().item() * (dt == torch.bfloat16)
        assert (out.cpu().double() - want).abs().max().item() <= tol
    # twice in a row: the same again
    out2 = torch.empty(M, I, device=DEV, dtype=torch.float32)
    ops.gemm(to_dev(a), to_dev(w), out2, silu_mul=True)
    assert torch.equal(out2, out)


@pytest.mark.parametrize("M,N,K", [(2100, 14000, 160), (1024, 28672, 128), (2048, 16384, 2048), (4000, 7200, 352),
                                   (2049, 14080, 128 + 32), (2048, 6144, 128),
                                   # 192 and 384 tiles, the last column tile partly outside
                                   (2048, 6000, 192), (4096, 6096, 160),
                                   # two and three row tiles, on either side of where they begin
                                   (256, 24576, 160), (257, 24576, 160), (513, 16384, 128)])
@pytest.mark.parametrize("mode", ["bf16", "f32", "f32+", "silu"])
def test_gemm_bf16_large_products_through_the_lds_ring(M, N, K, mode):
    """Products of a thousand rows and more with some hundred 256 x 256 tiles take the kernel whose operands go
    from memory straight into a ring of LDS buffers: rows and columns that do not fill the last tiles, k-steps
    from the ring's depth upwards, every epilogue; twice in a row gives the same bits."""
    from glassbox_amd import ops
    a, w = rnd(M, K, seed=11).bfloat16(), rnd(N, K, seed=12).bfloat16()
    if mode == "silu":
        a, w = a * 0.25, w * 0.25
    full = a.double() @ w.double().T
    c0 = rnd(M, N, seed=13)
    if mode == "silu":
        g, u = full[:, :N // 2], full[:, N // 2:]
        want = g / (1 + torch.exp(-g)) * u
    else:
        want = full + (c0.double() if mode == "f32+" else 0)
    outs = []
    for _ in range(2):
        if mode == "silu":
            c = torch.full((M, N // 2), 7.0, device=DEV, dtype=torch.bfloat16)
        else:
            c = to_dev(c0.clone(), torch.bfloat16 if mode == "bf16" else torch.float32)
        ops.gemm(to_dev(a), to_dev(w), c, accumulate=(mode == "f32+"), silu_mul=(mode == "silu"))
        outs.append(c)
    tol = 1e-4 * math.sqrt(K) + (2 ** -8) * want.abs().max().item() * (mode in ("bf16", "silu"))
    assert (outs[0].cpu().double() - want).abs().max().item() <= tol
    assert torch.equal(outs[0], outs[1])


@pytest.mark.parametrize("M,N,K", [
    # tiles of 256 and 224 rows, 224 and 192, 192 and 160, 160 and 128; one row in the last 32; a last column tile partly outside
    (1185, 11200, 640), (1601, 8112, 160), (641, 28672, 160), (705, 16320, 640), (1185, 16320, 160), (1313, 11200, 640)])
@pytest.mark.parametrize("mode", ["bf16", "f32", "f32+", "silu"])
def test_gemm_bf16_ring_with_tiles_of_two_heights(M, N, K, mode):
    """Rows dealt to tiles of fewer than 256 rows, every epilogue: the last row of each tile and the first of the next among
    those compared, and rows of C beyond the product left alone."""
    from glassbox_amd import ops
    lib = ops._lib("gemm_bf16")
    epi = {"bf16": 0, "f32": 0, "f32+": 1, "silu": 2}[mode]
    assert lib.gb_gemm_bf16_route(M, N, K, epi, 0, 0) == 1
    a, w = rnd(M, K, seed=11).bfloat16() * 0.25, rnd(N, K, seed=12).bfloat16() * 0.25
    full = a.float() @ w.float().T
    c0 = rnd(M, N, seed=13)
    cols = N // 2 if mode == "silu" else N
    want = full + c0 if mode == "f32+" else full
    if mode == "silu":
        g, u = full[:, :cols], full[:, cols:]
        want = g / (1 + torch.exp(-g)) * u
    room = torch.full((M + 40, cols), 7.0, device=DEV, dtype=torch.bfloat16 if mode in ("bf16", "silu") else torch.float32)
    if mode == "f32+":
        room[:M] = to_dev(c0)
    ops.gemm(to_dev(a), to_dev(w), room[:M], accumulate=(mode == "f32+"), silu_mul=(mode == "silu"))
    # sums of K products in 32-bit on either side, and the result's rounding
    tol = 1e-5 * math.sqrt(K) + (2 ** -8) * want.abs().max().item() * (mode in ("bf16", "silu"))
    assert (room[:M].cpu().float() - want).abs().max().item() <= tol
    assert bool((room[M:] == 7.0).all())


@pytest.mark.parametrize("mode", ["bf16", "f32", "f32+", "silu"])
@pytest.mark.parametrize("pad,shift", [(8, 0), (2, 0), (6, 2), (0, 4)])
def test_gemm_bf16_ring_writes_rows_that_are_no_whole_words(mode, pad, shift):
    """Rows of C that are longer than the product's, or begin between 16-byte words: the ring kernel's results are those
    it writes into a dense C, to the bit, and nothing beside them is written."""
    from glassbox_amd import ops
    M, N, K = 1030, 14000, 160
    a, w = to_dev(rnd(M, K, seed=11).bfloat16() * 0.25), to_dev(rnd(N, K, seed=12).bfloat16() * 0.25)
    cols = N // 2 if mode == "silu" else N
    dtype = torch.bfloat16 if mode in ("bf16", "silu") else torch.float32
    dense = torch.full((M, cols), 0.5, device=DEV, dtype=dtype)
    ops.gemm(a, w, dense, accumulate=(mode == "f32+"), silu_mul=(mode == "silu"))
    room = torch.full((M * (cols + pad) + shift,), 0.5, device=DEV, dtype=dtype)
    c = room[shift:].view(M, cols + pad)
    ops.gemm(a, w, c[:, :cols], accumulate=(mode == "f32+"), silu_mul=(mode == "silu"))
    assert torch.equal(c[:, :cols], dense)
    assert bool((c[:, cols:] == 0.5).all()) and bool((room[:shift] == 0.5).all())


@pytest.mark.parametrize("mode", ["bf16", "f32", "f32+", "silu"])
@pytest.mark.parametrize("over", [8, 16, 72, 120, 128, 136, 200, 248, 6, 130])
def test_gemm_bf16_ring_writes_the_last_columns_alike_by_words_and_one_by_one(mode, over):
    """Column tiles that C ends in: written four columns a lane, and, where rows of C are no words, one at a time."""
    from glassbox_amd import ops
    M, cols, K = (2050, 6912 + (over + 7) // 8 * 8, 128) if mode == "silu" else (1030, 13824 + over, 128)
    N = 2 * cols if mode == "silu" else cols
    assert ops.gemm_route(M, N, K, silu_mul=mode == "silu", accumulate=mode == "f32+") == "ring"
    a, w = to_dev(rnd(M, K, seed=11).bfloat16() * 0.25), to_dev(rnd(N, K, seed=12).bfloat16() * 0.25)
    dtype = torch.bfloat16 if mode in ("bf16", "silu") else torch.float32
    got = []
    for pad in ((-cols) % 8, (-cols) % 8 + 1):
        c = torch.full((M + 1, cols + pad), 0.5, device=DEV, dtype=dtype)
        ops.gemm(a, w, c[:M, :cols], accumulate=(mode == "f32+"), silu_mul=(mode == "silu"))
        assert bool((c[:, cols:] == 0.5).all()) and bool((c[M:] == 0.5).all())
        got.append(c[:M, :cols].clone())
    assert torch.equal(*got)
    rows = [0, 255, 256, M - 1]
    want = a[rows].double() @ w.double().T
    if mode == "silu":
        want = torch.nn.functional.silu(want[:, :cols]) * want[:, cols:]
    want = want + (0.5 if mode == "f32+" else 0)
    # sums of K products in 32-bit, and the result's rounding
    tol = 1e-5 * math.sqrt(K) + (2 ** -8) * want.abs().max().item() * (mode in ("bf16", "silu"))
    assert (got[0][rows].double() - want).abs().max().item() <= tol


@pytest.mark.parametrize("M", [5, 300, 1600])
def test_gemm_bf16_gated_unit_at_the_ends_of_its_range(M):
    """silu(gate) * up where the exponential or its reciprocal leaves the range, in the kernels that form it in their
    epilogue (few rows, tiles, the ring): the formula's own values in 32-bit, infinities among them."""
    from glassbox_amd import ops
    I, K = 4096, 128
    gates = torch.tensor([-3e38, -1e30, -200.0, -89.0, -88.0, -80.0, -1.0, -0.0, 0.0, 1e-30, 1.0, 80.0, 200.0, 1e30, float("inf"),
                          float("-inf")]).bfloat16()
    a, w = torch.zeros(M, K), torch.zeros(2 * I, K)
    a[:, 0], w[:I, 0], w[I:, 0] = 1.0, gates.float().repeat(I // len(gates) + 1)[:I], 1.0
    out = torch.full((M, I), 7.0, device=DEV, dtype=torch.bfloat16)
    ops.gemm(to_dev(a.bfloat16()), to_dev(w.bfloat16()), out, silu_mul=True)
    g = w[:I, 0].double()
    want = (g / (1 + torch.exp(-g)))[None, :].expand(M, I)
    got = out.cpu().double()
    assert torch.equal(torch.isnan(got), torch.isnan(want)) and torch.equal(torch.isinf(got), torch.isinf(want))
    fine = torch.isfinite(want)
    # a bfloat16 result; where exp(-gate) leaves the 32-bit range (2^128, from -gate = 88.8 on) the formula in 32-bit is zero,
    # which is at most 89 / 2^128 < 2^-121 off
    assert ((got - want).abs()[fine] <= 2 ** -8 * want.abs()[fine] + 2.0 ** -121).all()


@pytest.mark.parametrize("M", [5, 100, 300, 1600])
@pytest.mark.parametrize("clamped", [False, True])
def test_gemm_bf16_gated_unit_of_large_gates(M, clamped):
    """Gates up to the largest a bfloat16 holds, beside an up of 0 among others: silu(gate) is the gate itself there, and
    nothing on the way to it may leave the range (few rows, blocks, tiles, the ring; the clamped unit with a limit that no
    gate reaches)."""
    from glassbox_amd import ops
    I, K = 4096, 128
    gates = torch.tensor([2.0 ** 123, 2.0 ** 124, 2.2e37, 2.0 ** 127, 3e38, -3e38, 1e30]).bfloat16().float()
    ups = torch.tensor([1.0, 0.0, -1.0, 2.0 ** -60]).float()
    a, w = torch.zeros(M, K), torch.zeros(2 * I, K)
    a[:, 0], w[:I, 0], w[I:, 0] = 1.0, gates.repeat(I // len(gates) + 1)[:I], ups.repeat(I // len(ups))
    out = torch.full((M, I), 7.0, device=DEV, dtype=torch.bfloat16)
    if clamped:
        ops.gemm_glu(to_dev(a.bfloat16()), to_dev(w.bfloat16()), out, 3.2e38, 1.0, 0.0)
    else:
        ops.gemm(to_dev(a.bfloat16()), to_dev(w.bfloat16()), out, silu_mul=True)
    g, u = w[:I, 0], w[I:, 0]
    want = (g / (1 + torch.exp(-g)) * u)[None, :].expand(M, I).double()
    assert torch.isfinite(want).all()
    assert ((out.cpu().double() - want).abs() <= 2 ** -8 * want.abs()).all()


def test_gemm_bf16_gated_unit_rounds_alike_by_every_route():
    """One row of float32 results with SiLU-multiply, alone and among so many rows that the block kernel, the tiles, the
    ring or slices of k take the product: the sums are exact (one nonzero k), so what the unit makes of them is the same to
    the bit."""
    from glassbox_amd import ops
    I, K = 4096, 128
    w = torch.zeros(2 * I, K)
    w[:, 0] = rnd(2 * I, seed=31) * 3
    w = to_dev(w.bfloat16())
    rows = {}
    for M in (1, 5, 40, 100, 200, 300, 1600):
        a = torch.zeros(M, K, device=DEV, dtype=torch.bfloat16)
        a[:, 0] = 1.0
        out = torch.full((M, I), 7.0, device=DEV)
        ops.gemm(a, w, out, silu_mul=True)
        rows[M] = out.cpu()
    wide, K = torch.zeros(2 * I, 4096, device=DEV, dtype=torch.bfloat16), 4096
    wide[:, 0] = w[:, 0]
    wide, few = wide[:2048].contiguous(), 1024          # the first gates, and the second thousand of them as their ups
    for M in (5, 40, 200):
        a = torch.zeros(M, K, device=DEV, dtype=torch.bfloat16)
        a[:, 0] = 1.0
        out = torch.full((M, few), 7.0, device=DEV)
        ws = torch.empty(max(1, ops.gemm_split_floats(M, 2 * few, K)), device=DEV)
        ops.gemm(a, wide, out, silu_mul=True, workspace=ws)
        rows["divided", M] = out.cpu()
    for key, out in rows.items():
        assert torch.equal(out, (rows["divided", 5] if isinstance(key, tuple) else rows[1])[:1].expand_as(out)), key


@pytest.mark.parametrize("N,K,M,silu", [(96, 64, 1, False), (6144, 2048, 8, False), (352, 176, 5, True),
                                        (16384, 2048, 8, True), (480, 80, 33, False), (512, 4104, 64, True)])
@pytest.mark.parametrize("gamma_dtype", [torch.float32, torch.bfloat16])
def test_gemm_bf16_fused_rms_norm(N, K, M, silu, gamma_dtype):
    """The product that norms its float32 rows on the way, against norm-then-product in float64
    (crates/glassbox-core/src/model.rs:94-100 and 260 / 335)."""
    from glassbox_amd import ops
    x = rnd(M, K, seed=1, scale=3.0).float()
    x[0] *= 1e-3                                              # a row where eps matters
    g = (rnd(K, seed=2) * 0.3 + 1.0).to(gamma_dtype)
    w = (rnd(N, K, seed=3) / math.sqrt(K)).bfloat16()
    eps = 1e-5
    h = g.double() * (x.double() * torch.rsqrt(x.double().pow(2).mean(-1, keepdim=True) + eps))
    prod = h @ w.double().T
    if silu:
        gate, up = prod[:, :N // 2], prod[:, N // 2:]
        want = gate / (1 + torch.exp(-gate)) * up
    else:
        want = prod
    out = torch.full(want.shape, 9.0, device=DEV, dtype=torch.bfloat16)
    ops.gemm(to_dev(x), to_dev(w), out, silu_mul=silu, rms=(to_dev(g), eps))
    # bf16(g * x) as the operand: one rounding per element, 2^-9 relative, averaged over k
    tol = (2 ** -7) * want.abs().max().item() + 1e-3
    assert (out.cpu().double() - want).abs().max().item() <= tol
    # the unfused pair of kernels rounds elsewhere (bf16(g * x * s) as the operand) and is as close
    hn = torch.empty(M, K, device=DEV, dtype=torch.bfloat16)
    ops.rmsnorm(to_dev(x), to_dev(g), eps, hn)
    two = torch.empty_like(out)
    ops.gemm(hn, to_dev(w), two, silu_mul=silu)
    assert (two.cpu().double() - want).abs().max().item() <= tol


@pytest.mark.parametrize("M,N,K,N2,silu", [(1, 64, 176, 96, False), (5, 352, 64, 176, True), (8, 2048, 2048, 6144, False),
                                           (8, 2048, 8192, 16384, True), (3, 960, 2560, 2880, False),
                                           # more than 8 rows (tiles of 8 columns while they are few, of 16 beyond), and more than 16: the
                                           # skinny kernel emits and takes the partial sums of up to 64
                                           (12, 960, 2560, 2880, False), (40, 24704, 128, 512, False), (64, 352, 64, 176, True),
                                           (20, 4096, 1024, 1024, True), (9, 72, 264, 48, False), (17, 2048, 1024, 16384, True),
                                           (20, 960, 960, 5120, True), (33, 960, 776, 1600, False),
                                           # a k beyond 2,048: half tiles of up to 24 rows and of more, one tile, two
                                           (20, 968, 2056, 256, False), (32, 968, 2056, 256, False), (32, 5128, 2304, 256, False),
                                           (24, 6160, 2568, 256, False), (33, 24704, 2056, 256, False),
                                           # up to 16 rows, sums of 16 columns: two tiles a workgroup, of a number that two does not divide, and
                                           # four; four waves of two blocks and of three, eight of two, three and four
                                           (5, 4096, 512, 256, False), (12, 4096, 512, 256, False), (16, 8200, 264, 256, False), (5, 8216, 520, 256, False),
                                           (5, 8192, 520, 256, False), (9, 4104, 2632, 256, False), (9, 4104, 776, 256, True), (16, 8200, 1032, 256, False),
                                           (16, 4096, 2048, 256, False)])
@pytest.mark.parametrize("gamma_dtype", [torch.float32, torch.bfloat16])
def test_gemm_bf16_prepares_the_next_norm(M, N, K, N2, silu, gamma_dtype):
    """The product that adds into the residual and, on its way out, writes what the RMS norm that reads
    the residual next would compute (bf16(gamma * r) and partial sums of r^2), and the product that takes
    those: against norm-then-product in float64 (crates/glassbox-core/src/model.rs:94-100, 323-335)."""
    from glassbox_amd import ops
    parts_n = ops.gemm_emit_parts(M, N)
    assert parts_n == (-(-N // 8) if -(-N // 16) < 256 else -(-N // 16)) and ops.gemm_emit_mode(M, N, K) == 1
    stride = ops.parts_stride(M)
    assert stride == (8 if M <= 8 else 64)
    a, w = rnd(M, K, seed=1).bfloat16(), (rnd(N, K, seed=2) / math.sqrt(K)).bfloat16()
    r0 = rnd(M, N, seed=3, scale=2.0).float()
    g = (rnd(N, seed=4) * 0.3 + 1.0).to(gamma_dtype)
    eps = 1e-5
    plain = to_dev(r0.clone())
    ops.gemm(to_dev(a), to_dev(w), plain, accumulate=True)
    res, h = to_dev(r0.clone()), torch.zeros(M, N, device=DEV, dtype=torch.bfloat16)
    parts = torch.full((parts_n, stride), 7.0, device=DEV)
    ops.gemm(to_dev(a), to_dev(w), res, accumulate=True, emit=(to_dev(g), h, parts))
    assert torch.equal(res, plain)                                        # the residual is what it was without
    assert torch.equal(h, (to_dev(g).float() * res).bfloat16())
    ss = res.double().pow(2).sum(-1).cpu()
    assert ((parts[:, :M].double().sum(0).cpu() - ss).abs() <= 1e-5 * ss).all()
    assert ((parts[:, M:] == 0) | (parts[:, M:] == 7.0)).all()                # rows that do not exist: zero or untouched
    # the product that follows
    w2 = (rnd(N2, N, seed=5) / math.sqrt(N)).bfloat16()
    x = res.double().cpu()
    normed = g.double() * (x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + eps))
    prod = normed @ w2.double().T
    want = prod if not silu else prod[:, :N2 // 2] / (1 + torch.exp(-prod[:, :N2 // 2])) * prod[:, N2 // 2:]
    out = torch.full(want.shape, 9.0, device=DEV, dtype=torch.bfloat16)
    ops.gemm(h, to_dev(w2), out, silu_mul=silu, rms_parts=(parts, parts_n, eps))
    tol = (2 ** -7) * want.abs().max().item() + 1e-3                      # as for the norm computed on the way in
    assert (out.cpu().double() - want).abs().max().item() <= tol
    again = torch.empty_like(out)
    ops.gemm(res, to_dev(w2), again, silu_mul=silu, rms=(to_dev(g), eps))
    assert ((out.float() - again.float()).abs() <= 2 ** -6 * (1 + again.float().abs())).all()


@pytest.mark.parametrize("N,K", [
    # one tile, part of one, and the last workgroup's tiles beyond the rows of W; k of a part of a block, of whole blocks, of a part
    # of a turn: four waves of two and three blocks, eight of two, four and five, sixteen of four and eight, and more turns than one
    (8, 8), (4, 64), (20, 520), (9, 776), (264, 1000), (2056, 1032), (40, 2048), (72, 2104), (136, 2568), (88, 4096), (48, 8200),
    # two, three and four tiles a workgroup, the last one's beyond the rows of W
    (4100, 584), (4104, 2632), (6148, 264), (6152, 2056), (8204, 968), (8216, 2112)])
@pytest.mark.parametrize("M", [1, 8, 9, 16])
def test_gemm_bf16_of_up_to_16_rows(M, N, K):
    """The products of a decode step against float64, and what one row holds stays its own: a row of A and a row of W
    that are not finite touch their row and their column of the result alone (the two k ranges of a tile stand side by side)."""
    from glassbox_amd import ops
    a, w = rnd(M, K, seed=1).bfloat16(), (rnd(N, K, seed=2) / math.sqrt(K)).bfloat16()
    da, dw = to_dev(a), to_dev(w)
    want = a.double() @ w.double().T
    c = torch.full((M, N), 9.0, device=DEV)
    ops.gemm(da, dw, c)
    tol = 1e-4    # 32-bit sums of products of numbers of variance 1 / K: 2^-24 sqrt(K) terms at most, K <= 8,200
    assert (c.cpu().double() - want).abs().max().item() <= tol
    if N >= 16:
        half = N // 16 * 8
        act = torch.full((M, half), 9.0, device=DEV, dtype=torch.bfloat16)
        ops.gemm(da, dw[:2 * half], act, silu_mul=True)
        g, u = want[:, :half], want[:, half:2 * half]
        unit = g / (1 + torch.exp(-g)) * u
        assert (act.cpu().double() - unit).abs().max().item() <= 2 ** -8 * unit.abs().max().item() + 10 * tol
    wild_a, wild_w = a.clone(), w.clone()
    wild_a[M - 1, K - 1], wild_w[N - 1, 0] = float("nan"), float("inf")
    ops.gemm(to_dev(wild_a), to_dev(wild_w), c)
    finite = torch.isfinite(c.cpu())
    assert finite[:M - 1, :N - 1].all() and not finite[M - 1].any() and not finite[:, N - 1].any()


@pytest.mark.parametrize("M,N,K", [(2048, 2048, 8192), (128, 2048, 2048), (40, 1008, 4104), (300, 960, 2560), (64, 2048, 8192)])
@pytest.mark.parametrize("gamma_dtype", [torch.float32, torch.bfloat16])
def test_gemm_bf16_that_divides_k_does_the_next_norm(M, N, K, gamma_dtype):
    """An accumulating product that divides k over workgroups adds its slices row by row, and with a row in hand
    writes the RMS norm of the new residual too: the rows the norm's own kernel would give."""
    from glassbox_amd import ops
    assert ops.gemm_emit_mode(M, N, K) == 2 and ops.gemm_emit_mode(4, N, K) != 2
    a, w = (rnd(M, K, seed=21) * 0.5).bfloat16(), (rnd(N, K, seed=22) * 0.1).bfloat16()
    res0, g = rnd(M, N, seed=23).float(), (rnd(N, seed=24) * 0.3 + 1).to(gamma_dtype)
    eps = 1e-5
    ws = torch.empty(ops.gemm_split_floats(M, N, K), device=DEV)
    res, h = to_dev(res0.clone()), torch.full((M, N), 9.0, device=DEV, dtype=torch.bfloat16)
    ops.gemm(to_dev(a), to_dev(w), res, accumulate=True, emit=(to_dev(g), h, eps), workspace=ws)
    want_res = res0.double() + a.double() @ w.double().T
    assert (res.cpu().double() - want_res).abs().max().item() <= 1e-4 * math.sqrt(K)
    # the residual is the same as without the norm, bit for bit; the rows are those of the norm's kernel but for
    # the order of its sum (a unit in the last place of bfloat16 at most)
    plain = to_dev(res0.clone())
    ops.gemm(to_dev(a), to_dev(w), plain, accumulate=True, workspace=ws)
    assert torch.equal(res, plain)
    normed = torch.empty_like(h)
    ops.rmsnorm(res, to_dev(g), eps, normed)
    assert ((h.float() - normed.float()).abs() <= 2 ** -7 * normed.float().abs() + 1e-6).all()
    x = res.cpu().double()
    want = g.double() * x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)
    assert (h.cpu().double() - want).abs().max().item() <= 2 ** -8 * want.abs().max().item() + 1e-6
    with pytest.raises(ops.KernelError, match="norm"):
        ops.gemm(to_dev(a), to_dev(w), res, accumulate=True, emit=(to_dev(g), h, eps))       # no workspace


@pytest.mark.parametrize("M,N,K", [(17, 4096, 14336), (24, 4096, 4160), (33, 576, 1536), (20, 96, 8192), (64, 72, 1088), (49, 8192, 1024),
                                   (64, 4088, 16384), (32, 8, 4096)])
def test_gemm_bf16_of_few_rows_that_divides_k_does_the_next_norm(M, N, K):
    """17 to 64 rows: slices of one to sixteen, some of them short; rows of two words a thread, of a few words in all."""
    test_gemm_bf16_that_divides_k_does_the_next_norm(M, N, K, torch.float32)


@pytest.mark.parametrize("M,N,K", [(17, 96, 4096), (33, 2048, 2048), (64, 2048, 8192), (100, 2048, 4160),
                                   # few tiles of a long k (Llama-3-8B's O and down projections)
                                   (96, 4096, 8192), (128, 4096, 4096),
                                   # 65 to 128 rows by many rows of W: from a k above 8,192 on
                                   (96, 6160, 8256), (65, 8192, 9216),
                                   # beyond 64 rows a slice of a long k keeps 1,024 of it
                                   (192, 2048, 4096), (256, 1024, 8192),
                                   # a k that is no multiple of 64: the tiled kernel's slices
                                   (200, 528, 8200), (40, 1008, 4104),
                                   # a thousand rows and more: slices of k through the 256 x 256 tiles
                                   (2048, 2048, 8192), (1100, 1008, 4160), (1024, 528, 5120),
                                   # and some hundred rows, rows and columns that no tile divides: on either side of where a k of
                                   # 8,192 is long enough, where few rows of a longer one are, and on the far side of 256 and 1,023
                                   (549, 528, 8192), (550, 528, 8192), (611, 1040, 8192), (320, 528, 14336), (257, 528, 17536),
                                   (1023, 528, 4416),
                                   # some hundred rows, a k of 2,048 and very few tiles
                                   (128, 2048, 2048), (300, 1008, 2112), (256, 1024, 2048)])
@pytest.mark.parametrize("mode", ["bf16", "f32", "f32+", "silu"])
def test_gemm_bf16_divides_k_over_workgroups(M, N, K, mode):
    """With a workspace, a product of few tiles has several workgroups a tile, each over a slice of k,
    and a second kernel adds their sums in a fixed order and applies the epilogue: against float64, and
    the same bits on every run."""
    from glassbox_amd import ops
    floats = ops.gemm_split_floats(M, N, K)
    assert floats > 0 and floats % (M * N) == 0 and floats // (M * N) >= 2
    a, w = rnd(M, K, seed=1).bfloat16(), (rnd(N, K, seed=2) / math.sqrt(K)).bfloat16()
    c0 = rnd(M, N, seed=3)
    prod = a.double() @ w.double().T
    if mode == "silu":
        want = prod[:, :N // 2] / (1 + torch.exp(-prod[:, :N // 2])) * prod[:, N // 2:]
    else:
        want = prod + (c0.double() if mode == "f32+" else 0)
    ws = torch.full((floats + 3,), float("nan"), device=DEV)[:floats]
    outs = []
    for _ in range(2):
        if mode == "silu":
            c = torch.full((M, N // 2), 7.0, device=DEV, dtype=torch.bfloat16)
        else:
            c = to_dev(c0.clone(), torch.bfloat16 if mode == "bf16" else torch.float32)
        ops.gemm(to_dev(a), to_dev(w), c, accumulate=(mode == "f32+"), silu_mul=(mode == "silu"), workspace=ws)
        outs.append(c)
    tol = 1e-4 * math.sqrt(K) + (2 ** -8) * want.abs().max().item() * (mode in ("bf16", "silu"))
    assert (outs[0].cpu().double() - want).abs().max().item() <= tol
    assert torch.equal(outs[0], outs[1])
    with pytest.raises(ops.KernelError, match="workspace"):
        ops.gemm(to_dev(a), to_dev(w), outs[0], accumulate=(mode == "f32+"), silu_mul=(mode == "silu"), workspace=ws[:8])


@pytest.mark.parametrize("M,N,K", [(65, 6144, 2048), (128, 16384, 2048), (96, 6144, 8192),
                                   # one, two, three k-steps, and seventeen
                                   (100, 4096, 64), (128, 4128, 128), (100, 5000, 192), (70, 6200, 1024), (128, 8200, 1088),
                                   # very many columns, a short k
                                   (128, 24600, 320), (96, 32760, 512),
                                   # 17 to 64 rows by very many rows of W and a short k: the wide tiles, not the skinny kernel
                                   (64, 49152, 256), (40, 33000, 192), (20, 40000, 192),
                                   # a narrow model's products: few tiles and a k too short to divide
                                   (96, 2560, 960), (200, 5120, 960), (256, 2500, 448), (129, 2100, 128)])
@pytest.mark.parametrize("mode", ["bf16", "f32", "f32+", "silu"])
def test_gemm_bf16_streams_products_of_some_hundred_rows(M, N, K, mode):
    """65 to 128 rows (to 256 in a narrow model), a k that is a multiple of 64, or a vocabulary at up to 64 rows: the block and the tiled
    kernel and, for the last, the held one, without slices of k (with or without a workspace on offer).
    Against float64, the same bits on every run, rows and columns beyond the last tile's edge untouched."""
    from glassbox_amd import ops
    if mode == "silu" and N % 16:
        N -= N % 16
    assert ops.gemm_split_floats(M, N, K) == 0
    a, w = rnd(M, K, seed=1).bfloat16(), (rnd(N, K, seed=2) / math.sqrt(K)).bfloat16()
    c0 = rnd(M, N, seed=3)
    prod = a.double() @ w.double().T
    if mode == "silu":
        want = prod[:, :N // 2] / (1 + torch.exp(-prod[:, :N // 2])) * prod[:, N // 2:]
    else:
        want = prod + (c0.double() if mode == "f32+" else 0)
    cols = want.shape[1]
    outs = []
    for _ in range(2):
        # a frame of untouched cells around the result: two more rows, a longer row stride
        dtype = torch.float32 if mode in ("f32", "f32+") else torch.bfloat16
        frame = torch.full((M + 2, cols + 8), 7.0, device=DEV, dtype=dtype)
        c = frame[:M, :cols]
        if mode == "f32+":
            c.copy_(to_dev(c0))
        ops.gemm(to_dev(a), to_dev(w), c, accumulate=(mode == "f32+"), silu_mul=(mode == "silu"))
        assert (frame[M:] == 7.0).all() and (frame[:, cols:] == 7.0).all()
        outs.append(c.clone())
    tol = 1e-4 * math.sqrt(K) + (2 ** -8) * want.abs().max().item() * (mode in ("bf16", "silu"))
    assert (outs[0].cpu().double() - want).abs().max().item() <= tol
    assert torch.equal(outs[0], outs[1])


@pytest.mark.parametrize("M,N,K", [(66, 1040, 1024), (131, 6144, 2048), (131, 16384, 512), (200, 5120, 960), (224, 1600, 2048), (300, 6160, 1088),
                                   (420, 16384, 576), (512, 6144, 2048), (611, 5120, 960), (1000, 5120, 960), (257, 2064, 4160), (64, 28672, 4096)])
@pytest.mark.parametrize("mode", ["bf16", "f32", "f32+", "silu", "workspace"])
def test_gemm_bf16_blocks_of_some_hundred_rows(M, N, K, mode):
    """Tiles of 64 to 256 rows by 64 to 128 rows of W, several k-steps on their way: fewer k-steps than that, rows and columns that no
    tile divides, with a workspace on offer; against float64, the same bits on every run, nothing beyond the last row and column."""
    from glassbox_amd import ops
    a, w = rnd(M, K, seed=1).bfloat16(), (rnd(N, K, seed=2) / math.sqrt(K)).bfloat16()
    c0 = rnd(M, N, seed=3).float()
    prod = (to_dev(a).double() @ to_dev(w).double().T)
    want = prod
    if mode == "silu":
        want = prod[:, :N // 2] / (1 + torch.exp(-prod[:, :N // 2])) * prod[:, N // 2:]
    elif mode == "f32+":
        want = prod + to_dev(c0).double()
    cols = want.shape[1]
    ws = torch.empty(max(1, ops.gemm_split_floats(M, N, K)), device=DEV) if mode == "workspace" else None
    outs = []
    for _ in range(2):
        frame = torch.full((M + 2, cols + 8), 7.0, device=DEV, dtype=torch.float32 if mode in ("f32", "f32+") else torch.bfloat16)
        c = frame[:M, :cols]
        if mode == "f32+":
            c.copy_(to_dev(c0))
        ops.gemm(to_dev(a), to_dev(w), c, accumulate=(mode == "f32+"), silu_mul=(mode == "silu"), workspace=ws)
        assert (frame[M:] == 7.0).all() and (frame[:, cols:] == 7.0).all()
        outs.append(c.clone())
    # a float32 sum of K products of 16-bit numbers, and the rounding of the result to 16 bits
    tol = 1e-4 * math.sqrt(K) + (2 ** -8) * want.abs().max().item() * (mode in ("bf16", "silu", "workspace"))
    assert (outs[0].double() - want).abs().max().item() <= tol
    assert torch.equal(outs[0], outs[1])


# sizes that the held kernel takes in every mode below (a storing product of 160 to 255 tiles of 16 rows of W, or a long k), at the edges of
# its registers, rings and tiles: column blocks of rows, k-blocks a wave (none for some waves, the most), columns that no tile divides
HELD = [(17, 2576, 576), (32, 2600, 960), (33, 2564, 320), (48, 4072, 448), (49, 2568, 1088), (64, 2561, 1984), (24, 8240, 4096), (33, 12290, 2048),
        (17, 6152, 2112), (64, 5130, 1344), (31, 2050, 3136)]


@pytest.mark.parametrize("M,N,K", [(17, 2056, 64), (32, 2050, 576), (33, 2048, 960), (48, 8250, 1984), (49, 4112, 2048), (64, 5120, 960),
                                   # a wave's most blocks of k; tiles that do not divide among the workgroups; a short k and few tiles
                                   (31, 33000, 448), (20, 976, 128), (64, 960, 704)] + HELD)
@pytest.mark.parametrize("mode", ["bf16", "f32", "silu", "silu_f32", "parts", "parts_f32", "padded"])
def test_gemm_bf16_holds_the_rows_and_streams_w(M, N, K, mode):
    """17 to 64 rows by many rows of W, held in the registers of a workgroup for every compute unit (HELD; the others lie on either side
    of where that pays): against the product in float64, alone, with the gated unit, behind the partial sums of a norm, and into
    rows that are no whole words."""
    from glassbox_amd import ops
    held = (M, N, K) in HELD
    if mode[:4] in ("silu", "part"):
        N -= N % 16
    parts = 75 if mode.startswith("parts") else 0
    if held and mode in ("bf16", "f32", "padded"):
        assert ops.gemm_route(M, N, K) == "held"
    check_held(M, N, K, silu=mode.startswith("silu") or (parts > 0 and N % 32 == 0), n_parts=parts, f32=mode.endswith("f32") or mode == "padded",
               padded=mode == "padded")


@pytest.mark.parametrize("M,N,K,silu", [(17, 16384, 3072, True), (32, 6160, 3072, False), (64, 5120, 960, True), (49, 960, 64, True), (33, 5120, 576, True),
                                        (53, 6144, 2048, False)])
@pytest.mark.parametrize("n", [255, 256, 257, 384, 511])
def test_gemm_bf16_held_rows_behind_many_partial_sums(M, N, K, silu, n):
    """Partial sums of a norm up to and beyond the 256 that the held kernel asks for at once (a row of 3,072 leaves 384)."""
    from glassbox_amd import ops
    assert ops.gemm_route(M, N, K, silu_mul=silu, parts=True) == "held"
    check_held(M, N, K, silu=silu, n_parts=n, f32=True, padded=False)


@pytest.mark.parametrize("M,N,K,n", [
    # a k of up to 2,048, beyond with one tile a workgroup and up to 32 rows, and beyond; as many partial sums as are asked for at once,
    # up to eight more a lane, and several rounds of eight; k of whole turns and of part of one
    (33, 1600, 2040, 255), (40, 1600, 2056, 256), (17, 4096, 5120, 320), (24, 1280, 8192, 640), (32, 6160, 5120, 511), (33, 6160, 2056, 129),
    (48, 2576, 3072, 384), (64, 6160, 3080, 1025), (17, 6160, 4104, 130),
    # half a tile a workgroup: up to 24 rows, and up to 32 of a short k and of a longer one
    (24, 968, 2560, 0), (25, 968, 2560, 0), (32, 1000, 2048, 0)])
@pytest.mark.parametrize("silu", [False, True])
def test_gemm_bf16_of_17_to_64_rows_of_a_short_and_of_a_long_k(M, N, K, n, silu):
    """The kernel that streams W through all of a workgroup's waves in both of its forms, against float64."""
    from glassbox_amd import ops
    N -= N % 16 if silu else 0
    assert ops.gemm_route(M, N, K, silu_mul=silu, parts=n > 0) == "few"
    check_held(M, N, K, silu=silu, n_parts=n, f32=True, padded=False)


@pytest.mark.parametrize("M,K", [(1, 64), (8, 2048), (9, 776), (16, 2048), (20, 960), (48, 2048)])
@pytest.mark.parametrize("off", [1, 2, 3])
def test_gemm_bf16_takes_partial_sums_anywhere(M, K, off):
    """Partial sums are floats of the caller's, also where they are no 16-byte words: a view that begins some floats on gives the bits of
    a tensor of its own, in a product and in the rotating one."""
    from glassbox_amd import ops
    nh, nkv, hd, n, eps, stride = 4, 2, 32, 75, 1e-5, ops.parts_stride(M)
    a, w = to_dev(rnd(M, K, seed=1).bfloat16()), to_dev((rnd((nh + 2 * nkv) * hd, K, seed=2) / math.sqrt(K)).bfloat16())
    room = to_dev(torch.rand(n * stride + off, generator=torch.Generator().manual_seed(off)) * 20 + 0.1)
    outs = [[], []]
    for out, parts in zip(outs, (room[off:], room[off:].clone())):
        c = torch.empty(M, w.shape[0], device=DEV)
        ops.gemm(a, w, c, rms_parts=(parts, n, eps))
        qkv = torch.empty(M, w.shape[0], device=DEV, dtype=torch.bfloat16)
        ops.gemm_rope(a, w, qkv, nh, nkv, hd, None, None, None, None, None, rms_parts=(parts, n, eps))
        out += [c.cpu(), qkv.cpu()]
    assert torch.equal(outs[0][0], outs[1][0]) and torch.equal(outs[0][1], outs[1][1])
    scale = 1 / torch.sqrt(room[off:].cpu().double().view(n, stride)[:, :M].sum(0) / K + eps)
    want = a.cpu().double() @ w.cpu().double().T * scale.unsqueeze(1)
    assert ((outs[0][0].double() - want).abs() <= sum_bound(a.cpu(), w.cpu()) * scale.max().item() + 2 ** -21 * want.abs()).all()


def sum_bound(a, w):
    """What a float32 sum of products of 16-bit numbers may be off by: sqrt(K) roundings' worth of 2^-24 of a partial sum, which is
    about the product of the rows' lengths at most; eight times that."""
    K = a.shape[1]
    return 8 * 2 ** -24 * math.sqrt(K) * a.double().norm(dim=1).max().item() * w.double().norm(dim=1).max().item()


def check_held(M, N, K, silu, n_parts, f32, padded):
    from glassbox_amd import ops
    a, w = rnd(M, K, seed=M).bfloat16(), (rnd(N, K, seed=N) / math.sqrt(K)).bfloat16()
    prod, tol, parts, scale = a.double() @ w.double().T, sum_bound(a, w), None, None
    if n_parts:
        eps = 1e-5
        sums = rnd(n_parts, 64, seed=5).abs().float() * (75 / n_parts) + 0.1
        scale = 1 / torch.sqrt(sums[:, :M].double().sum(0) / K + eps)
        prod, tol = prod * scale.unsqueeze(1), tol * scale.max().item()
        parts = (to_dev(sums), n_parts, eps)
    want = prod
    bound = torch.full_like(prod, tol) + 2 ** -21 * prod.abs()      # (the scale: a few roundings of 2^-24)
    if silu:
        g, u = prod[:, :N // 2], prod[:, N // 2:]
        want = g / (1 + torch.exp(-g)) * u
        # |d silu / dg| < 1.1, |silu(g)| <= |g|; the unit's own arithmetic a few roundings
        bound = bound[:, :N // 2] * 1.1 * u.abs() + bound[:, N // 2:] * g.abs() + tol * tol * 1.1 + 2 ** -20 * want.abs()
    cols = want.shape[1]
    room = torch.full((M, cols + 3), 7.0, device=DEV, dtype=torch.float32 if f32 else torch.bfloat16)
    out = room[:, 1:cols + 1] if padded else room.view(-1)[:M * cols].view(M, cols)
    ops.gemm(to_dev(a), to_dev(w), out, silu_mul=silu, rms_parts=parts)
    if not f32:
        bound = bound * 1.01 + 2 ** -8 * want.abs()
    assert ((out.cpu().double() - want).abs() <= bound).all()
    if padded:
        assert (room[:, 0] == 7.0).all() and (room[:, cols + 1:] == 7.0).all()
    again = torch.empty_like(out)
    ops.gemm(to_dev(a), to_dev(w), again, silu_mul=silu, rms_parts=parts)
    assert torch.equal(out, again)
    # a row's bits do not depend on the rows beside it
    if M > 33:
        few = torch.empty(M - 1, cols, device=DEV, dtype=out.dtype)
        if (M - 1 + 15) // 16 == (M + 15) // 16:   # (as many column blocks: the same kernel)
            ops.gemm(to_dev(a[1:]), to_dev(w), few, silu_mul=silu,
                     rms_parts=None if parts is None else (to_dev(torch.cat([parts[0].cpu()[:, 1:], parts[0].cpu()[:, :1]], 1)), *parts[1:]))
            assert torch.equal(few, out[1:])


def test_gemm_bf16_split_k_is_the_same_on_every_run():
    from glassbox_amd import ops
    a, w = to_dev(rnd(8, 8192, seed=1).bfloat16()), to_dev(rnd(2048, 8192, seed=2).bfloat16())
    base = torch.zeros(8, 2048, device=DEV)
    ops.gemm(a, w, base, accumulate=True)
    for _ in range(5):
        again = torch.zeros(8, 2048, device=DEV)
        ops.gemm(a, w, again, accumulate=True)
        assert torch.equal(again, base)


def test_gemm_bf16_one_hot_rows_and_columns():
    """Every (row, column, k) lands where it should: W picks single columns of A."""
    from glassbox_amd import ops
    M, K, N = 150, 136, 200
    a = rnd(M, K, seed=5).bfloat16()
    w = torch.zeros(N, K)
    for n in range(N):
        w[n, (7 * n + 3) % K] = 1.0
    c = torch.zeros(M, N, device=DEV)
    ops.gemm(to_dev(a), to_dev(w.bfloat16()), c)
    want = a.float()[:, [(7 * n + 3) % K for n in range(N)]]
    assert torch.equal(c.cpu(), want)
    for rows in (17, 9, 8, 5, 1):   # the skinny kernel, and the one that folds two k ranges into a tile
        c2 = torch.zeros(rows, N, device=DEV)
        ops.gemm(to_dev(a[:rows]), to_dev(w.bfloat16()), c2)
        assert torch.equal(c2.cpu(), want[:rows]), rows


def test_gemm_refuses_bad_inner_size():
    from glassbox_amd import ops
    a, w = torch.zeros(4, 12, device=DEV, dtype=torch.bfloat16), torch.zeros(8, 12, device=DEV, dtype=torch.bfloat16)
    with pytest.raises(ops.KernelError, match="multiple of 8"):
        ops.gemm(a, w, torch.zeros(4, 8, device=DEV, dtype=torch.bfloat16))


# -------------------------------------------------------------------- elementwise
@pytest.mark.parametrize("n,d", [(1, 7), (3, 100), (5, 576), (2, 1537), (4, 2048)])
@pytest.mark.parametrize("out_dtype", [torch.float32, torch.bfloat16])
def test_rmsnorm(n, d, out_dtype):
    from glassbox_amd import ops
    x, g, eps = rnd(n, d, seed=1, scale=3.0), rnd(d, seed=2) + 1.0, 3e-5
    want = g.double() * (x.double() * torch.rsqrt(x.double().pow(2).mean(-1, keepdim=True) + eps))
    out = torch.empty(n, d, device=DEV, dtype=out_dtype)
    ops.rmsnorm(to_dev(x), to_dev(g), eps, out)
    tol = 1e-5 if out_dtype == torch.float32 else 2 ** -8
    assert ((out.cpu().double() - want).abs() <= tol * (1 + want.abs())).all()
    # picked rows
    rows = torch.tensor([n - 1, 0], dtype=torch.int32, device=DEV)
    out2 = torch.empty(2, d, device=DEV, dtype=out_dtype)
    ops.rmsnorm(to_dev(x), to_dev(g), eps, out2, rows)
    assert torch.equal(out2.cpu(), out.cpu()[[n - 1, 0]])


def test_embed():
    from glassbox_amd import ops
    table = rnd(37, 50, seed=1)
    ids = torch.tensor([5, 0, 36, 5], dtype=torch.int32, device=DEV)
    for dt in (torch.float32, torch.bfloat16):
        out = torch.empty(4, 50, device=DEV)
        ops.embed(to_dev(table, dt), ids, out)
        assert torch.equal(out.cpu(), table.to(dt).float()[[5, 0, 36, 5]])


def test_silu_mul():
    from glassbox_amd import ops
    gu = rnd(6, 2 * 173, seed=4, scale=4.0)
    g, u = gu[:, :173].double(), gu[:, 173:].double()
    want = g / (1 + torch.exp(-g)) * u
    out = torch.empty(6, 173, device=DEV)
    ops.silu_mul(to_dev(gu), out)
    assert (out.cpu().double() - want).abs().max().item() < 1e-5


@pytest.mark.parametrize("hd,theta", [(16, 10000.0), (48, 500000.0), (128, 130000.0), (80, 10000.0),
                                      (10, 10000.0)])   # 10: no multiple of 4, the kernel that goes pair by pair
def test_rope_table_and_rotation(hd, theta):
    """Against the plain implementation: pairing (i, i + hd/2), sign, 32-bit angle at long positions."""
    from glassbox_amd import ops
    from glassbox_amd.parts.rotary import Rotary
    from plain import llama
    pos = [0, 1, 17, 4095, 100003]
    n, nh, nkv = len(pos), 3, 2
    rot = Rotary(hd, theta)
    cos = torch.empty(n, hd // 2, device=DEV)
    sin = torch.empty_like(cos)
    ops.rope_table(torch.tensor(pos, dtype=torch.int32, device=DEV), torch.from_numpy(rot.inv_host).to(DEV), cos, sin)
    s_want, c_want = llama.rope_angles(pos, hd, theta)
    assert np.abs(cos.cpu().numpy() - c_want).max() < 1e-7 and np.abs(sin.cpu().numpy() - s_want).max() < 1e-7
    qkv = rnd(n, (nh + 2 * nkv) * hd, seed=3)
    page = 16
    k_pages = torch.zeros(ops.key_pages_shape(4, nkv, page, hd), device=DEV)
    v_pages = torch.zeros(4, nkv, hd, page, device=DEV)
    slots = torch.tensor([3, 16 + 15, 32, 0, 63], dtype=torch.int32, device=DEV)
    buf = to_dev(qkv.clone())
    ops.rope_store(buf, cos, sin, slots, k_pages, v_pages, nh, nkv, hd)
    q_want = llama.rope(qkv[:, :nh * hd].double().reshape(n, nh, hd), pos, theta)
    k_want = llama.rope(qkv[:, nh * hd:(nh + nkv) * hd].double().reshape(n, nkv, hd), pos, theta)
    got_q = buf.cpu()[:, :nh * hd].double().reshape(n, nh, hd)
    assert (got_q - q_want).abs().max().item() < 1e-5
    assert torch.equal(got_q[0], qkv[0, :nh * hd].double().reshape(nh, hd)), "position 0 must leave the vector as it is"
    for i, s in enumerate(slots.tolist()):
        got_k = ops.unpack_keys(k_pages)[s // page, :, s % page, :].cpu().double()
        got_v = v_pages[s // page, :, :, s % page].cpu()
        assert (got_k - k_want[i]).abs().max().item() < 1e-5
        assert torch.equal(got_v, qkv[i, (nh + nkv) * hd:].reshape(nkv, hd))


ROPE_PRODUCTS = [(1, 4, 2, 16, 64), (8, 3, 1, 32, 96), (5, 6, 2, 48, 80), (8, 32, 32, 64, 2048), (33, 8, 2, 128, 264),
                 (64, 15, 5, 64, 960), (7, 4, 0, 32, 64),
                 # 432 and 400 tiles of 8 pairs: a tile and a half to a workgroup, and two tiles each
                 (40, 50, 2, 128, 128), (20, 48, 1, 128, 192)]


@pytest.mark.parametrize("nh,nkv,hd,page", [(4, 2, 16, 16), (32, 32, 64, 16), (5, 1, 48, 32), (8, 2, 128, 16), (3, 3, 80, 64)])
def test_rope_store_in_bfloat16_moves_whole_pieces(nh, nkv, hd, page):
    """bfloat16 rows of head sizes in steps of 16 (a lane takes 8 dimensions and their partners): rotated queries
    in the row, rotated keys in the row and in their pages, values in theirs, against float64
    (crates/glassbox-core/src/model.rs:102-115, 273-275)."""
    from glassbox_amd import ops
    from plain import llama
    n, theta = 37, 130000.0
    g = torch.Generator().manual_seed(hd)
    pos = torch.randint(0, 6000, (n,), generator=g).tolist()
    s64, c64 = llama.rope_angles(pos, hd, theta)
    cos, sin = to_dev(torch.from_numpy(c64).float()), to_dev(torch.from_numpy(s64).float())
    qkv = rnd(n, (nh + 2 * nkv) * hd, seed=7).bfloat16()
    pages = 4
    slots = torch.randperm(pages * page, generator=g)[:n].to(torch.int32)
    k_pages = torch.zeros(ops.key_pages_shape(pages, nkv, page, hd), device=DEV, dtype=torch.bfloat16)
    v_pages = torch.zeros(pages, nkv, hd, page, device=DEV, dtype=torch.bfloat16)
    buf = to_dev(qkv.clone())
    ops.rope_store(buf, cos, sin, to_dev(slots), k_pages, v_pages, nh, nkv, hd)
    q_want = llama.rope(qkv[:, :nh * hd].double().reshape(n, nh, hd), pos, theta)
    k_want = llama.rope(qkv[:, nh * hd:(nh + nkv) * hd].double().reshape(n, nkv, hd), pos, theta)
    got = buf.cpu()
    tol = 2 ** -8 * 1.5 * qkv.abs().max().item()   # one rounding to bfloat16 of a value up to sqrt(2) times the largest input
    assert (got[:, :nh * hd].double().reshape(n, nh, hd) - q_want).abs().max().item() <= tol
    assert (got[:, nh * hd:(nh + nkv) * hd].double().reshape(n, nkv, hd) - k_want).abs().max().item() <= tol
    assert torch.equal(got[:, (nh + nkv) * hd:], qkv[:, (nh + nkv) * hd:]), "values stay as they are"
    idx = slots.long()
    assert torch.equal(ops.unpack_keys(k_pages).cpu()[idx // page, :, idx % page, :], got[:, nh * hd:(nh + nkv) * hd].reshape(n, nkv, hd))
    assert torch.equal(v_pages.cpu()[idx // page, :, :, idx % page], qkv[:, (nh + nkv) * hd:].reshape(n, nkv, hd))
    free = torch.ones(pages * page, dtype=torch.bool)
    free[idx] = False
    fi = torch.nonzero(free).flatten()
    assert ops.unpack_keys(k_pages).cpu()[fi // page, :, fi % page, :].abs().sum().item() == 0
    assert v_pages.cpu()[fi // page, :, :, fi % page].abs().sum().item() == 0


@pytest.mark.parametrize("M,nh,nkv,hd,K,normed", [p + (False,) for p in ROPE_PRODUCTS] +
                         [p + (True,) for p in ROPE_PRODUCTS if p[0] <= 16])   # the norm on the way in serves 16 rows
def test_gemm_bf16_rotates_and_writes_the_cache(M, nh, nkv, hd, K, normed):
    """The stacked q/k/v product whose epilogue rotates query and key heads and writes keys and values into
    the pages: against the product, the rotation and the cache write in float64
    (crates/glassbox-core/src/model.rs:260-276), and against the two kernels it replaces."""
    from glassbox_amd import ops
    from plain import llama
    page, N = 16, (nh + 2 * nkv) * hd
    g = torch.Generator().manual_seed(M + hd)
    x = rnd(M, K, seed=1, scale=2.0).float()
    gamma, eps = (rnd(K, seed=2) * 0.3 + 1.0).float(), 1e-5
    w = (rnd(N, K, seed=3) / math.sqrt(K)).bfloat16()
    pos = torch.randint(0, 5000, (M,), generator=g).tolist()
    theta = 130000.0
    s64, c64 = llama.rope_angles(pos, hd, theta)
    cos, sin = to_dev(torch.from_numpy(c64).float()), to_dev(torch.from_numpy(s64).float())
    slots = torch.randperm(4 * page, generator=g)[:M].to(torch.int32)
    if normed:
        a_dev = to_dev(x)
        h64 = gamma.double() * (x.double() * torch.rsqrt(x.double().pow(2).mean(-1, keepdim=True) + eps))
        rms = (to_dev(gamma), eps)
    else:
        a_dev = to_dev(x.bfloat16())
        h64 = x.bfloat16().double()
        rms = None
    prod = h64 @ w.double().T
    q_want = llama.rope(prod[:, :nh * hd].reshape(M, nh, hd), pos, theta).reshape(M, nh * hd)
    store = nkv > 0
    k_pages = torch.zeros(ops.key_pages_shape(4, max(nkv, 1), page, hd), device=DEV, dtype=torch.bfloat16)
    v_pages = torch.zeros(4, max(nkv, 1), hd, page, device=DEV, dtype=torch.bfloat16)
    qkv = torch.full((M, N), 9.0, device=DEV, dtype=torch.bfloat16)
    ops.gemm_rope(a_dev, to_dev(w), qkv, nh, nkv, hd, cos, sin, to_dev(slots) if store else None,
                  k_pages if store else None, v_pages if store else None, rms=rms)
    tol = (2 ** -7) * prod.abs().max().item() + 1e-3
    assert (qkv[:, :nh * hd].cpu().double() - q_want).abs().max().item() <= tol
    if store:
        k_want = llama.rope(prod[:, nh * hd:(nh + nkv) * hd].reshape(M, nkv, hd), pos, theta)
        v_want = prod[:, (nh + nkv) * hd:].reshape(M, nkv, hd)
        for i, sl in enumerate(slots.tolist()):
            assert (ops.unpack_keys(k_pages)[sl // page, :, sl % page, :].cpu().double() - k_want[i]).abs().max().item() <= tol
            assert (v_pages[sl // page, :, :, sl % page].cpu().double() - v_want[i]).abs().max().item() <= tol
        # the rows hold what the pages hold
        assert torch.equal(qkv[0, nh * hd:(nh + nkv) * hd].reshape(nkv, hd),
                           ops.unpack_keys(k_pages)[slots[0] // page, :, slots[0] % page, :])
        # the two kernels it replaces round once more (the product to bfloat16 before the rotation)
        two = torch.empty_like(qkv)
        ops.gemm(a_dev, to_dev(w), two, rms=rms)
        k2, v2 = torch.zeros_like(k_pages), torch.zeros_like(v_pages)
        ops.rope_store(two, cos, sin, to_dev(slots), k2, v2, nh, nkv, hd)
        # (a rotated value can be much smaller than the two it is made of, so the bound is absolute)
        assert (two.float() - qkv.float()).abs().max().item() <= 2 * tol
        assert (k2.float() - k_pages.float()).abs().max().item() <= 2 * tol
        assert (v2.float() - v_pages.float()).abs().max().item() <= 2 * tol


@pytest.mark.parametrize("M,nh,nkv,hd,K", [(17, 32, 32, 64, 2048), (24, 32, 8, 128, 4096), (64, 32, 32, 64, 2048), (33, 9, 3, 64, 576),
                                           (48, 31, 9, 48, 128), (32, 40, 0, 64, 1024), (19, 129, 1, 16, 64), (64, 60, 2, 64, 1984),
                                           (48, 31, 9, 48, 2048), (32, 40, 0, 64, 2048), (19, 131, 1, 16, 4096), (64, 60, 3, 64, 1984)])
def test_gemm_bf16_rotates_and_writes_the_cache_with_the_rows_held(M, nh, nkv, hd, K):
    """The same where a workgroup holds the rows and walks over several tiles of W (a wave then prepares one of them), and, of a short k,
    beside where it does."""
    from glassbox_amd import ops
    assert ops.gemm_route(M, (nh + 2 * nkv) * hd, K, heads=True) == ("few" if K in (64, 128, 1024) or nkv == 2 else "held")
    test_gemm_bf16_rotates_and_writes_the_cache(M, nh, nkv, hd, K, False)


@pytest.mark.parametrize("M,nh,nkv,hd,K,n,kernel", [
    (20, 9, 3, 64, 576, 72, "held"), (49, 9, 3, 64, 576, 72, "held"), (32, 32, 8, 96, 3072, 384, "held"), (24, 32, 8, 128, 4096, 256, "held"),
    (64, 32, 32, 64, 2048, 257, "held"), (33, 32, 8, 48, 2048, 511, "held"), (17, 24, 8, 64, 512, 64, "few"), (8, 9, 3, 64, 576, 72, "few"),
    (40, 15, 5, 64, 960, 120, "few"),
    # a longer k than 2,048: a tile and a half, one tile and two tiles a workgroup
    (20, 72, 12, 64, 5120, 320, "few"), (24, 8, 4, 64, 2304, 300, "few"), (40, 15, 5, 64, 2560, 160, "few"), (64, 32, 8, 128, 4096, 256, "few"),
    (24, 50, 2, 128, 5120, 320, "few")])
def test_gemm_bf16_rotates_behind_the_partial_sums_of_a_norm(M, nh, nkv, hd, K, n, kernel):
    """The stacked q/k/v product of rows whose norm comes as partial sums: the scale is in what is rotated, in the rows and in both
    pages.  Against float64, element by element."""
    from glassbox_amd import ops
    assert ops.gemm_route(M, (nh + 2 * nkv) * hd, K, heads=True, parts=True) == kernel
    check_rotation(M, nh, nkv, hd, K, n, 16)


# one tile a workgroup, two, three and four, with each number of waves and blocks that few_plan (csrc/hip/gemm_bf16.hip) gives them; the
# last workgroup's tiles beyond the rows of W, k of whole turns and of part of one; pages that are a power of two and pages that are not
@pytest.mark.parametrize("M,nh,nkv,hd,K,n,page", [
    (9, 4, 2, 16, 72, 0, 48), (16, 32, 16, 64, 520, 64, 16), (12, 15, 5, 64, 776, 97, 48), (16, 64, 16, 64, 704, 0, 64), (9, 96, 16, 64, 640, 80, 48),
    (16, 8, 4, 48, 1032, 0, 80), (9, 48, 8, 64, 1000, 125, 16), (12, 32, 32, 64, 1032, 129, 48), (16, 96, 16, 64, 1000, 0, 16),
    (9, 8, 2, 128, 2568, 321, 48), (16, 48, 8, 64, 2600, 0, 32), (12, 32, 8, 128, 4096, 256, 16), (9, 8, 4, 64, 2048, 256, 48),
    (16, 40, 12, 64, 2048, 0, 16), (12, 32, 32, 64, 2048, 256, 48), (12, 32, 32, 64, 2048, 0, 16), (16, 50, 1, 80, 448, 56, 48),
    (8, 96, 16, 64, 1536, 192, 48), (5, 32, 32, 64, 2048, 256, 80), (8, 97, 16, 64, 2048, 0, 16), (1, 8, 2, 128, 2560, 320, 48),
    (8, 8, 4, 16, 8192, 0, 48)])
def test_gemm_bf16_of_up_to_16_rows_rotates_and_writes_pages_of_any_size(M, nh, nkv, hd, K, n, page):
    check_rotation(M, nh, nkv, hd, K, n, page)


def check_rotation(M, nh, nkv, hd, K, n, page):
    """A rotating product, behind n partial sums of a norm or (n = 0) of rows as they are, against float64 element by element."""
    from glassbox_amd import ops
    N, eps = (nh + 2 * nkv) * hd, 1e-5
    g = torch.Generator().manual_seed(M + n)
    a, w = (rnd(M, K, seed=1) * 0.5).bfloat16(), (rnd(N, K, seed=2) / math.sqrt(K)).bfloat16()
    stride = ops.parts_stride(M)
    scale = torch.ones(M, dtype=torch.float64)
    if n:
        sums = torch.rand(n, stride, generator=g) * 20 + 0.1
        scale = 1 / torch.sqrt(sums[:, :M].double().sum(0) / K + eps)
    angles = torch.rand(M, hd // 2, generator=g) * 6
    cos, sin = angles.cos(), angles.sin()
    slots = torch.randperm(5 * page, generator=g)[:M].to(torch.int32)
    prod = ((a.double() @ w.double().T) * scale.unsqueeze(1)).view(M, nh + 2 * nkv, hd)
    lo, hi = prod[..., :hd // 2], prod[..., hd // 2:]
    c, s = cos.double().unsqueeze(1), sin.double().unsqueeze(1)
    want = torch.cat([lo * c - hi * s, hi * c + lo * s], -1)
    want[:, nh + nkv:] = prod[:, nh + nkv:]
    size = torch.cat([lo.abs() + hi.abs()] * 2, -1)
    bound = 2 * sum_bound(a, w) * scale.max().item() + 2 ** -21 * size + 2 ** -8 * want.abs()
    k_pages = torch.zeros(ops.key_pages_shape(5, nkv, page, hd), device=DEV, dtype=torch.bfloat16)
    v_pages = torch.zeros(5, nkv, hd, page, device=DEV, dtype=torch.bfloat16)
    qkv = torch.full((M, N), 9.0, device=DEV, dtype=torch.bfloat16)
    ops.gemm_rope(to_dev(a), to_dev(w), qkv, nh, nkv, hd, to_dev(cos), to_dev(sin), to_dev(slots), k_pages, v_pages, rms_parts=(to_dev(sums), n, eps) if n else None)
    rows = qkv.cpu().double().view(M, nh + 2 * nkv, hd)
    assert ((rows - want).abs() <= bound).all()
    keys, idx = ops.unpack_keys(k_pages).cpu().double(), slots.long()
    assert torch.equal(keys[idx // page, :, idx % page, :], rows[:, nh:nh + nkv])
    assert torch.equal(v_pages.cpu().double()[idx // page, :, :, idx % page], rows[:, nh + nkv:])
    free = torch.ones(5 * page, dtype=torch.bool)
    free[idx] = False
    idx = torch.nonzero(free).flatten()
    assert (keys[idx // page, :, idx % page, :] == 0).all() and (v_pages.cpu()[idx // page, :, :, idx % page] == 0).all()


@pytest.mark.parametrize("M", [1, 8, 9, 12, 16, 17])
@pytest.mark.parametrize("N,K", [(16, 8), (264, 520), (5120, 960), (8208, 2048), (16384, 1032)])
def test_gemm_bf16_clamped_unit_of_few_rows(M, N, K):
    """min(g, limit) sigmoid(alpha g) (clamp(u) + plus) at the limits' edges and inside them, against float64 element by element."""
    from glassbox_amd import ops
    a, w = (rnd(M, K, seed=1) * 3).bfloat16(), (rnd(N, K, seed=2) / math.sqrt(K)).bfloat16()
    limit, alpha, plus = 4.0, 1.702, 1.0
    prod, tol = a.double() @ w.double().T, sum_bound(a, w)
    g, u = prod[:, :N // 2].clamp(max=limit), prod[:, N // 2:].clamp(-limit, limit)
    want = g / (1 + torch.exp(-alpha * g)) * (u + plus)
    # |d (g sigmoid(alpha g)) / dg| < 1.1 and its size at most |g|; the unit's own arithmetic a few roundings; one to 16 bits
    bound = tol * (1.1 * (u + plus).abs() + g.abs()) + 1.1 * tol * tol + 2 ** -20 * (1 + want.abs()) + 2 ** -8 * want.abs()
    out = torch.full((M, N // 2), 9.0, device=DEV, dtype=torch.bfloat16)
    ops.gemm_glu(to_dev(a), to_dev(w), out, limit, alpha, plus)
    assert ((out.cpu().double() - want).abs() <= bound).all()


@pytest.mark.parametrize("M,K", [(1, 64), (8, 2048), (9, 72), (16, 1032), (20, 64), (48, 2048)])
@pytest.mark.parametrize("angles", [True, False])
def test_gemm_bf16_rotation_leaves_values_alone(M, K, angles):
    """A dimension of a value that is not finite stays that dimension's, in the row and in the page; and so does one of a query or a
    key where the call has no angles, while with angles it reaches the one that it is paired with and no other."""
    from glassbox_amd import ops
    nh, nkv, hd, page = 4, 2, 32, 16
    heads = nh + 2 * nkv
    a, w = rnd(M, K, seed=1).bfloat16(), (rnd(heads * hd, K, seed=2) / math.sqrt(K)).bfloat16()
    wild = [(1, 5), (nh + 1, hd // 2 + 3), (nh + nkv, 2), (nh + 2 * nkv - 1, hd - 1)]      # (head, dimension): query, key, two values
    want = torch.zeros(M, heads, hd, dtype=torch.bool)
    for (head, d), value in zip(wild, [float("inf"), float("nan"), float("inf"), float("nan")]):
        w[head * hd + d] = value
        want[:, head, d] = True
        if angles and head < nh + nkv:
            want[:, head, (d + hd // 2) % hd] = True
    turn = torch.rand(M, hd // 2, generator=torch.Generator().manual_seed(3)) * 6
    slots = torch.randperm(4 * page, generator=torch.Generator().manual_seed(4))[:M].to(torch.int32)
    k_pages = torch.zeros(ops.key_pages_shape(4, nkv, page, hd), device=DEV, dtype=torch.bfloat16)
    v_pages = torch.zeros(4, nkv, hd, page, device=DEV, dtype=torch.bfloat16)
    qkv = torch.full((M, heads * hd), 9.0, device=DEV, dtype=torch.bfloat16)
    ops.gemm_rope(to_dev(a), to_dev(w), qkv, nh, nkv, hd, to_dev(turn.cos()) if angles else None, to_dev(turn.sin()) if angles else None,
                  to_dev(slots), k_pages, v_pages)
    assert torch.equal(~torch.isfinite(qkv.cpu()).view(M, heads, hd), want)
    idx = slots.long()
    assert torch.equal(~torch.isfinite(ops.unpack_keys(k_pages).cpu())[idx // page, :, idx % page, :], want[:, nh:nh + nkv])
    assert torch.equal(~torch.isfinite(v_pages.cpu())[idx // page, :, :, idx % page], want[:, nh + nkv:])


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("hd,page", [(16, 16), (64, 16), (128, 32), (40, 16)])
def test_rope_store_writes_values_of_portions_in_tiles(dtype, hd, page):
    """Values of prompt portions go to the transposed pages sixteen positions at a time: the pages must
    come out as when every row is written by itself.  Portions that start in the middle of a page, end
    in the middle of one, are shorter than a page, and single rows before them."""
    from glassbox_amd import ops
    nh, nkv = 3, 2
    q_lens, pos0 = [1, 1, 40, 16, 7, 33], [9, 0, 5, 32, 0, 47]
    n, n_dec = sum(q_lens), 2
    q_start = np.concatenate([[0], np.cumsum(q_lens)[:-1]]).tolist()
    pages_of, slots, next_page = [], [], 0
    for length, first in zip(q_lens, pos0):                   # every request has pages of its own, in a scrambled order
        count = -(-(first + length) // page)
        mine = [next_page + (7 * i) % count for i in range(count)] if count % 7 else list(range(next_page, next_page + count))
        next_page += count
        pages_of.append(mine)
        slots += [mine[p // page] * page + p % page for p in range(first, first + length)]
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=DEV)
    qkv = rnd(n, (nh + 2 * nkv) * hd, seed=5).to(dtype)
    cos, sin = torch.rand(n, hd // 2, device=DEV), torch.rand(n, hd // 2, device=DEV)
    results = []
    for portions in (None, (n_dec, i32(q_start), i32(q_lens), i32(pos0), n_dec, len(q_lens) - n_dec, max(q_lens))):
        k_pages = torch.zeros(ops.key_pages_shape(next_page, nkv, page, hd), device=DEV, dtype=dtype)
        v_pages = torch.zeros(next_page, nkv, hd, page, device=DEV, dtype=dtype)
        buf = to_dev(qkv.clone())
        ops.rope_store(buf, cos, sin, i32(slots), k_pages, v_pages, nh, nkv, hd, portions=portions)
        results.append((buf.cpu(), k_pages.cpu(), v_pages.cpu()))
    for a, b in zip(*results):
        assert torch.equal(a, b)
    assert results[0][2].abs().sum() > 0


@pytest.mark.parametrize("nh,nkv,hd,page,q_lens,n_dec", [
    # one, four and two heads a lane; heads that a workgroup's lanes do not divide, and more lanes than heads are left
    (32, 32, 64, 16, [1] * 30 + [482], 30), (9, 3, 64, 16, [1, 1, 17, 40], 2), (5, 2, 48, 32, [33, 15], 0), (6, 3, 96, 16, [1, 700], 1),
    (32, 32, 64, 16, [1, 1023], 1), (34, 9, 64, 64, [777, 778], 0), (30, 5, 128, 16, [1100], 0), (40, 24, 16, 16, [1, 4200], 1),
    (30, 3, 32, 16, [4099], 0), (15, 5, 64, 16, [4097], 0)])
def test_rope_store_of_steps_with_portions_in_one_launch(nh, nkv, hd, page, q_lens, n_dec):
    """Rotation, key writes, values of single rows and of portions in one launch, against every row written by itself."""
    from glassbox_amd import ops
    pos0 = [(5 * i) % 23 + (9 if i < n_dec else 0) for i in range(len(q_lens))]
    n, slots, next_page = sum(q_lens), [], 0
    for length, first in zip(q_lens, pos0):
        count = -(-(first + length) // page)
        mine = [next_page + (7 * i) % count for i in range(count)] if count % 7 else list(range(next_page, next_page + count))
        next_page += count
        slots += [mine[p // page] * page + p % page for p in range(first, first + length)]
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=DEV)
    q_start = np.concatenate([[0], np.cumsum(q_lens)[:-1]]).tolist()
    qkv = rnd(n, (nh + 2 * nkv) * hd, seed=5).bfloat16()
    cos, sin = torch.rand(n, hd // 2, device=DEV), torch.rand(n, hd // 2, device=DEV)
    for rotate in (True, False):
        results = []
        for portions in (None, (n_dec, i32(q_start), i32(q_lens), i32(pos0), n_dec, len(q_lens) - n_dec, max(q_lens))):
            k_pages = torch.zeros(ops.key_pages_shape(next_page, nkv, page, hd), device=DEV, dtype=torch.bfloat16)
            v_pages = torch.zeros(next_page, nkv, hd, page, device=DEV, dtype=torch.bfloat16)
            buf = to_dev(qkv.clone())
            ops.rope_store(buf, cos, sin, i32(slots), k_pages, v_pages, nh, nkv, hd, rotate=rotate, portions=portions)
            results.append((buf, k_pages, v_pages))
        for a, b in zip(*results):
            assert torch.equal(a, b)
        assert results[0][2].abs().sum() > 0


# ---------------------------------------------------------------------- attention
def paged_setup(ctx_lens, nkv, hd, page, seed, dtype, scatter=True):
    """Keys and values of several requests scattered over pages in a shuffled order."""
    g = torch.Generator().manual_seed(seed)
    total_pages = sum(-(-c // page) for c in ctx_lens) + 3
    perm = torch.randperm(total_pages, generator=g).tolist() if scatter else list(range(total_pages))
    k_pages = torch.randn(total_pages, nkv, page, hd, generator=g).to(dtype)   # unowned slots hold junk
    v_pages = torch.randn(total_pages, nkv, hd, page, generator=g).to(dtype)   # values are kept transposed
    tables, ks, vs = [], [], []
    for c in ctx_lens:
        np_ = -(-c // page)
        t = [perm.pop() for _ in range(np_)]
        tables.append(t)
        k = torch.randn(c, nkv, hd, generator=g).to(dtype)
        v = torch.randn(c, nkv, hd, generator=g).to(dtype)
        for p in range(c):
            k_pages[t[p // page], :, p % page, :] = k[p]
            v_pages[t[p // page], :, :, p % page] = v[p]
        ks.append(k)
        vs.append(v)
    maxp = max(len(t) for t in tables)
    table_t = torch.tensor([t + [-1] * (maxp - len(t)) for t in tables], dtype=torch.int32)
    return k_pages, v_pages, table_t, ks, vs


def plain_attention_rows(q, ks, vs, tok_seq, positions, nh, scale, window):
    out = torch.zeros_like(q, dtype=torch.float64)
    n, _ = q.shape
    hd = ks[0].shape[-1]
    group = nh // ks[0].shape[1]
    for i in range(n):
        k, v, p = ks[tok_seq[i]].double(), vs[tok_seq[i]].double(), positions[i]
        lo = max(0, p - window + 1) if window else 0
        for h in range(nh):
            s = (k[lo:p + 1, h // group] @ q[i, h * hd:(h + 1) * hd].double()) * scale
            w = torch.softmax(s, 0)
            out[i, h * hd:(h + 1) * hd] = w @ v[lo:p + 1, h // group]
    return out


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("nh,nkv,hd,window", [(4, 2, 16, 0), (3, 1, 32, 0), (6, 2, 48, 0), (8, 8, 64, 0),
                                              (8, 2, 128, 0), (5, 5, 80, 0), (4, 2, 32, 37), (2, 1, 256, 0)])
def test_attention_plain_kernel(dtype, nh, nkv, hd, window):
    from glassbox_amd import ops
    page = 16
    ctx_lens = [1, 300, 77, 16, 530]
    k_pages, v_pages, tables, ks, vs = paged_setup(ctx_lens, nkv, hd, page, seed=hd + nh, dtype=dtype)
    # rows: the last token of every request, plus a portion in the middle of request 1 and the first tokens of 4
    tok_seq = [0, 1, 2, 3, 4] + [1] * 5 + [4] * 3
    positions = [c - 1 for c in ctx_lens] + [100, 101, 102, 103, 104] + [0, 1, 2]
    n = len(tok_seq)
    q = rnd(n, nh * hd, seed=11).to(dtype)
    scale = 1 / math.sqrt(hd)
    out = torch.empty(n, nh * hd, device=DEV, dtype=dtype)
    ops.attention_plain(to_dev(q), out, torch.tensor(positions, dtype=torch.int32, device=DEV),
                        torch.tensor(tok_seq, dtype=torch.int32, device=DEV), to_dev(tables), to_dev(ops.pack_keys(k_pages)),
                        to_dev(v_pages), nh, scale, window)
    want = plain_attention_rows(q, ks, vs, tok_seq, positions, nh, scale, window)
    tol = 2e-5 if dtype == torch.float32 else 2 ** -7
    err = (out.cpu().double() - want).abs().max().item()
    assert err < tol, err


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("nh,nkv,hd,window,page", [(4, 2, 16, 0, 16), (8, 8, 64, 0, 16), (3, 1, 32, 0, 48), (8, 2, 128, 0, 32),
                                                   (2, 1, 256, 0, 64), (4, 2, 32, 300, 16), (5, 5, 80, 0, 64)])
def test_attention_plain_spread_over_workgroups_gives_the_bits_of_one_workgroup(dtype, nh, nkv, hd, window, page):
    """With a workspace the plain kernel gives every chunk of 256 keys a workgroup and merges them in a second kernel,
    by the same steps in the same order as one workgroup that walks them: bit for bit the same rows, and those of the
    float64 formula.  Contexts of one chunk, of a chunk and a key, of many; a window that starts inside a page."""
    from glassbox_amd import ops
    ctx_lens = [1, 256, 257, 1200, 700]
    k_pages, v_pages, tables, ks, vs = paged_setup(ctx_lens, nkv, hd, page, seed=hd + nh + page, dtype=dtype)
    tok_seq = [0, 1, 2, 3, 4, 3, 3]
    positions = [c - 1 for c in ctx_lens] + [600, 255]
    n = len(tok_seq)
    q = rnd(n, nh * hd, seed=12).to(dtype)
    scale = 1 / math.sqrt(hd)
    args = (torch.tensor(positions, dtype=torch.int32, device=DEV), torch.tensor(tok_seq, dtype=torch.int32, device=DEV),
            to_dev(tables), to_dev(ops.pack_keys(k_pages)), to_dev(v_pages), nh, scale, window)
    walked = torch.empty(n, nh * hd, device=DEV, dtype=dtype)
    ops.attention_plain(to_dev(q), walked, *args)
    floats = ops.attention_plain_split_floats(n, nh, hd, page, 1280)
    assert floats > 0
    ws = torch.full((floats,), float("nan"), device=DEV)
    spread = torch.empty(n, nh * hd, device=DEV, dtype=dtype)
    ops.attention_plain(to_dev(q), spread, *args, workspace=ws, max_context=1280)
    assert torch.equal(spread, walked)
    want = plain_attention_rows(q, ks, vs, tok_seq, positions, nh, scale, window)
    tol = 2e-5 if dtype == torch.float32 else 2 ** -7
    assert (walked.cpu().double() - want).abs().max().item() < tol
    # many (token, head) pairs, or contexts of one chunk: nothing to spread
    assert ops.attention_plain_split_floats(2000, nh, hd, page, 1280) == 0
    assert ops.attention_plain_split_floats(n, nh, hd, page, 256) == 0
    with pytest.raises(ops.KernelError, match="workspace"):
        ops.attention_plain(to_dev(q), spread, *args, workspace=ws[:100], max_context=1280)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("nkv,hd", [(2, 64), (8, 32), (4, 16)])
def test_attention_plain_of_few_workgroups_and_of_more_gives_the_same_bits(dtype, nkv, hd):
    """32-bit launches of up to 2,048 workgroups over contexts of 33, 64 or 112 keys and more (up to 256, up to 640 and more workgroups), in
    one chunk or spread over workgroups, ask for a chunk's keys and values at once: chunks that end around a page and around 256 keys, on either side of each
    of these lines: the same bits, and those of the float64 formula."""
    from glassbox_amd import ops
    nh = 8
    ctx_lens = [1, 17, 191, 192, 193, 239, 240, 241, 255, 256, 257, 447, 448, 700]
    k_pages, v_pages, tables, ks, vs = paged_setup(ctx_lens, nkv, hd, 16, seed=hd + nkv, dtype=dtype)
    n = len(ctx_lens)
    q, scale = rnd(n, nh * hd, seed=12).to(dtype), 1 / math.sqrt(hd)
    rest = (to_dev(tables), to_dev(ops.pack_keys(k_pages)), to_dev(v_pages), nh, scale, 0)

    def rows(count, spread=False, longest=700, among=n):
        seq = [i % among for i in range(count)]
        pos = torch.tensor([ctx_lens[i] - 1 for i in seq], dtype=torch.int32, device=DEV)
        out = torch.full((count, nh * hd), 7.0, device=DEV, dtype=dtype)
        floats = ops.attention_plain_split_floats(count, nh, hd, 16, 700) if spread else 0
        more = dict(workspace=torch.full((floats,), float("nan"), device=DEV), max_context=700) if spread else dict(max_context=longest)
        ops.attention_plain(to_dev(q[seq]), out, pos, torch.tensor(seq, dtype=torch.int32, device=DEV), *rest, **more)
        return out.cpu()

    few = rows(n)
    for count, longest in ((10, 256), (10, 200), (10, 199), (n, 0)):    # (the first ten contexts are of up to 256 keys)
        assert torch.equal(rows(count, longest=longest), few[:count])
    # 256 and 264 workgroups, 640 and 648, 2,048 and 2,056; the longest context on either side of 33, 64 and 112 keys and of one chunk (one
    # that is longer than it was said to be is walked all the same)
    for count, longest in ((32, 32), (32, 33), (33, 33), (33, 63), (33, 64), (33, 257), (80, 64), (81, 64), (81, 111), (81, 112), (256, 256), (257, 256)):
        assert torch.equal(rows(count, longest=longest, among=10), few[[i % 10 for i in range(count)]])
    want = plain_attention_rows(q, ks, vs, list(range(n)), [c - 1 for c in ctx_lens], nh, scale, 0)
    assert (few.double() - want).abs().max().item() < (2e-5 if dtype == torch.float32 else 2 ** -7)
    for count in (n, 26, 27, 85, 86):       # three chunks each: 336, 624 and 648, 2,040 and 2,064
        assert torch.equal(rows(count, spread=True), few[[i % n for i in range(count)]])


@pytest.mark.parametrize("hd", [8, 16, 24, 40, 48, 56, 64])
def test_attention_plain_of_few_workgroups_gives_the_bits_of_the_walk(hd):
    """The kernel that asks for a chunk's keys and values at once (attention_plain_early_kernel), one workgroup a row and a
    workgroup a chunk: chunks that end around a page and around 256 keys, a cap and slopes and sinks; and a context that is longer
    than the launch was told.  The same bits as the walk (no longest context given)."""
    from glassbox_amd import ops
    nh, nkv = 6, 2
    ctx_lens = [1, 15, 16, 17, 64, 241, 255, 256, 257, 272, 511, 600]
    k_pages, v_pages, tables, ks, vs = paged_setup(ctx_lens, nkv, hd, 16, seed=hd, dtype=torch.float32)
    n, scale = len(ctx_lens), 1 / math.sqrt(hd)
    q, pos, seq = to_dev(rnd(n, nh * hd, seed=3)), torch.tensor([c - 1 for c in ctx_lens], dtype=torch.int32, device=DEV), \
        torch.arange(n, dtype=torch.int32, device=DEV)
    args = (pos, seq, to_dev(tables), to_dev(ops.pack_keys(k_pages)), to_dev(v_pages), nh, scale, 0)
    for more in ({}, dict(softcap=5.0), dict(slopes=to_dev(rnd(nh, seed=4).abs() * 0.1), sinks=to_dev(rnd(nh, seed=5)))):
        def out(**kw):
            o = torch.full((n, nh * hd), 7.0, device=DEV)
            ops.attention_plain(q, o, *args, **more, **kw)
            return o
        walk = out()
        floats = ops.attention_plain_split_floats(n, nh, hd, 16, 600)
        assert floats > 0
        assert torch.equal(out(max_context=256), walk)
        assert torch.equal(out(max_context=600, workspace=torch.full((floats,), float("nan"), device=DEV)), walk)
    want = plain_attention_rows(q.cpu(), ks, vs, list(range(n)), [c - 1 for c in ctx_lens], nh, scale, 0)
    o = torch.empty(n, nh * hd, device=DEV)
    ops.attention_plain(q, o, *args, max_context=256)
    assert (o.cpu().double() - want).abs().max().item() < 2e-5


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("nh,nkv,hd,page", [(4, 2, 16, 16), (8, 8, 64, 16), (3, 1, 32, 48), (2, 1, 128, 32), (2, 2, 256, 16),
                                            (5, 5, 80, 64)])
def test_attention_plain_eight_rows_a_workgroup_gives_the_bits_of_one_row_a_workgroup(dtype, nh, nkv, hd, page):
    """Many rows of prompt portions go eight rows a workgroup, which loads a key once where the eight are one request's
    consecutive tokens: bit for bit the rows of the one-row form.  Portions that start and end inside a group of
    eight, a group across the edge of a chunk of 256 keys (its first tokens have no key in the last chunk), single
    decoded tokens between portions; a head size and page for which the form is not built takes the one-row form."""
    from glassbox_amd import ops
    ctx_lens = [120, 263, 701, 531, 40]
    k_pages, v_pages, tables, ks, vs = paged_setup(ctx_lens, nkv, hd, page, seed=hd + nh + page + 1, dtype=dtype)
    rows = ([(0, p) for p in range(0, 101)]            # 101 rows: the next portion starts inside a group
            + [(1, p) for p in range(251, 262)]        # across key 256 in the middle of a group
            + [(2, 700)]                               # a decoded token
            + [(3, p) for p in range(509, 531)]        # across key 512
            + [(4, p) for p in range(0, 40)] + [(1, 262)])
    tok_seq, positions = [r[0] for r in rows], [r[1] for r in rows]
    n = len(rows)
    q = rnd(n, nh * hd, seed=14).to(dtype)
    scale = 1 / math.sqrt(hd)
    pos_d, seq_d = torch.tensor(positions, dtype=torch.int32, device=DEV), torch.tensor(tok_seq, dtype=torch.int32, device=DEV)
    rest = (to_dev(tables), to_dev(ops.pack_keys(k_pages)), to_dev(v_pages), nh, scale, 0)
    qd = to_dev(q)
    grouped = torch.empty(n, nh * hd, device=DEV, dtype=dtype)
    ops.attention_plain(qd, grouped, pos_d, seq_d, *rest, grouped=True)
    single = torch.empty(n, nh * hd, device=DEV, dtype=dtype)
    ops.attention_plain(qd, single, pos_d, seq_d, *rest)
    # the groups of eight fall elsewhere when the step's rows start at another row
    shifted = torch.empty(n, nh * hd, device=DEV, dtype=dtype)
    ops.attention_plain(qd[:3], shifted[:3], pos_d[:3], seq_d[:3], *rest, grouped=True)
    ops.attention_plain(qd[3:], shifted[3:], pos_d[3:], seq_d[3:], *rest, grouped=True)
    assert torch.equal(shifted, single)
    assert torch.equal(grouped, single)
    want = plain_attention_rows(q, ks, vs, tok_seq, positions, nh, scale, 0)
    tol = 2e-5 if dtype == torch.float32 else 2 ** -7
    assert (grouped.cpu().double() - want).abs().max().item() < tol


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_attention_finds_one_far_key(dtype):
    """One key among hundreds is made to stand out: the output must be its value, wherever it lies
    (first or last slot of a page, first page, a page far away)."""
    from glassbox_amd import ops
    nh, nkv, hd, page, ctx = 4, 2, 32, 16, 700
    k_pages, v_pages, tables, ks, vs = paged_setup([ctx], nkv, hd, page, seed=1, dtype=dtype)
    q = rnd(1, nh * hd, seed=2).to(dtype)
    for target in (0, 15, 16, 255, 256, 511, 683, 699):
        kp = k_pages.clone()
        for kvh in range(nkv):
            # the key at `target` points along the mean query of its group, scaled up
            qg = q[0].float().reshape(nh, hd)[kvh * 2:(kvh + 1) * 2]
            key = torch.stack([qg[0], qg[1]]).mean(0)
            # make both heads of the group agree on the direction: use head 0's query for both
            kp[tables[0, target // page], kvh, target % page, :] = (qg[0] * 40).to(dtype)
        qq = q.clone().float().reshape(nh, hd)
        qq[1::2] = qq[0::2]   # both heads of a group ask the same
        qq = qq.reshape(1, nh * hd).to(dtype)
        out = torch.empty(1, nh * hd, device=DEV, dtype=dtype)
        ops.attention_plain(to_dev(qq), out, torch.tensor([ctx - 1], dtype=torch.int32, device=DEV),
                            torch.tensor([0], dtype=torch.int32, device=DEV), to_dev(tables), to_dev(ops.pack_keys(kp)),
                            to_dev(v_pages), nh, 1 / math.sqrt(hd), 0)
        want = vs[0][target].float().repeat_interleave(2, 0).reshape(-1)
        assert (out.cpu().float()[0] - want).abs().max().item() < 2e-2, f"key at {target} was not found"


class BareContext:
    """What the tuned attention bindings read from a step's context, for a hand-made batch: single-token
    requests first, then portions."""

    def __init__(self, q_lens, ctx_lens, tables, max_context=None):
        from types import SimpleNamespace
        self.num_seqs = len(q_lens)
        n_dec = sum(1 for l in q_lens if l == 1)
        assert all(l == 1 for l in q_lens[:n_dec]) and all(l > 1 for l in q_lens[n_dec:])
        q_start = np.concatenate([[0], np.cumsum(q_lens)[:-1]]).tolist()
        pos0 = [c - l for c, l in zip(ctx_lens, q_lens)]
        self.tok_seq = [s for s, l in enumerate(q_lens) for _ in range(l)]
        self.pos_list = [pos0[s] + j for s, l in enumerate(q_lens) for j in range(l)]
        i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=DEV)
        self.positions, self.q_start, self.q_len, self.pos0 = i32(self.pos_list), i32(q_start), i32(q_lens), i32(pos0)
        self.tables = [to_dev(tables)]
        self.host = {"n_decode": n_dec, "max_q_len": max(q_lens), "max_context": max_context or max(ctx_lens)}
        self._bufs = {}

    def buffer(self, name, shape, dtype):
        return self._bufs.setdefault((name, tuple(shape)), torch.empty(shape, dtype=dtype, device=DEV))


@pytest.mark.parametrize("nh,nkv,hd,window", [(4, 2, 16, 0), (3, 1, 32, 0), (6, 2, 48, 0), (8, 8, 64, 0), (8, 2, 128, 0),
                                              (6, 3, 96, 0), (4, 4, 112, 0), (4, 2, 128, 70),
                                              (16, 1, 64, 0), (5, 5, 80, 0), (4, 2, 64, 37), (4, 4, 64, 300), (2, 1, 112, 0)])
@pytest.mark.parametrize("page", [16, 64])
def test_tuned_attention_against_the_plain_kernel(nh, nkv, hd, window, page):
    """The matrix-core kernels for decoding and for prompt portions against their plain twin and the
    float64 formula: contexts that end at every offset of a page, chunks that split, windows."""
    from types import SimpleNamespace
    from glassbox_amd import ops
    q_lens = [1, 1, 1, 1, 1, 5, 70, 16, 130]
    ctx_lens = [1, 17, 256, 700, 1025, 5, 300, 16, 530]      # portions 5/5, 70 ending at 300, 16/16, 130 ending at 530
    k_pages, v_pages, tables, ks, vs = paged_setup(ctx_lens, nkv, hd, page, seed=hd + nh, dtype=torch.bfloat16)
    ctx = BareContext(q_lens, ctx_lens, tables, max_context=1100)
    n = sum(q_lens)
    q = (rnd(n, nh * hd, seed=11) * 0.7).bfloat16()
    scale = 1 / math.sqrt(hd)
    cache = SimpleNamespace(k_pages=to_dev(ops.pack_keys(k_pages)), v_pages=to_dev(v_pages), group=0)
    assert ops.tuned_attention_supports(cache.k_pages, nh, window)
    out = torch.zeros(n, nh * hd, device=DEV, dtype=torch.bfloat16)
    qd = to_dev(q)
    ops.attention_decode(qd, out, ctx, cache, nh, scale, window)
    ops.attention_prefill(qd, out, ctx, cache, nh, scale, window)
    twin = torch.zeros_like(out)
    ops.attention_plain(qd, twin, ctx.positions, torch.tensor(ctx.tok_seq, dtype=torch.int32, device=DEV), ctx.tables[0],
                        cache.k_pages, cache.v_pages, nh, scale, window)
    want = plain_attention_rows(q, ks, vs, ctx.tok_seq, ctx.pos_list, nh, scale, window)
    err = (out.cpu().double() - want).abs().max(dim=1).values
    bad = torch.nonzero(err > 2 ** -6).flatten().tolist()
    assert not bad, f"rows {bad[:8]} (request, position) {[(ctx.tok_seq[i], ctx.pos_list[i]) for i in bad[:8]]}: {err[bad[:8]]}"
    # both are roundings to bfloat16 of nearly equal 32-bit results: at most a unit or two in the last place apart
    assert ((out.float() - twin.float()).abs() <= 2 ** -7 * (1 + twin.float().abs())).all()


@pytest.mark.parametrize("nh,nkv,hd,window", [(4, 2, 16, 0), (8, 8, 64, 0), (6, 3, 96, 0), (8, 2, 128, 70), (4, 4, 64, 300), (32, 16, 32, 0)])
def test_tuned_attention_with_32_bit_result_rows(nh, nkv, hd, window):
    """The same kernels writing float32 rows (for a caller that goes on in 32-bit, like the difference of two heads):
    the softmax weights then enter the value product in two bfloat16 parts, so the rows are the float64 formula's on
    the bfloat16 operands to a few units of the 16th bit, not of the 8th; single tokens, short and long portions, chunks
    that split."""
    from types import SimpleNamespace
    from glassbox_amd import ops
    q_lens = [1, 1, 1, 1, 1, 5, 70, 16, 1101]
    ctx_lens = [1, 17, 256, 700, 1025, 5, 300, 16, 1303]
    k_pages, v_pages, tables, ks, vs = paged_setup(ctx_lens, nkv, hd, 16, seed=hd + nh, dtype=torch.bfloat16)
    ctx = BareContext(q_lens, ctx_lens, tables, max_context=1400)
    n = sum(q_lens)
    q = (rnd(n, nh * hd, seed=11) * 0.7).bfloat16()
    scale = 1 / math.sqrt(hd)
    cache = SimpleNamespace(k_pages=to_dev(ops.pack_keys(k_pages)), v_pages=to_dev(v_pages), group=0)
    out = torch.full((n, nh * hd + 4), 7.0, device=DEV, dtype=torch.float32)[:, :nh * hd]   # rows wider than the heads
    qd = to_dev(q)
    ops.attention_decode(qd, out, ctx, cache, nh, scale, window)
    ops.attention_prefill(qd, out, ctx, cache, nh, scale, window)
    want = plain_attention_rows(q, ks, vs, ctx.tok_seq, ctx.pos_list, nh, scale, window)
    err = (out.cpu().double() - want).abs().max(dim=1).values
    bad = torch.nonzero(err > 2e-4 * (1 + want.abs().max())).flatten().tolist()
    assert not bad, f"rows {bad[:8]} (request, position) {[(ctx.tok_seq[i], ctx.pos_list[i]) for i in bad[:8]]}: {err[bad[:8]]}"
    narrow = torch.zeros(n, nh * hd, device=DEV, dtype=torch.bfloat16)
    ops.attention_decode(qd, narrow, ctx, cache, nh, scale, window)
    ops.attention_prefill(qd, narrow, ctx, cache, nh, scale, window)
    assert ((out - narrow.float()).abs() <= 2 ** -6 * (1 + out.abs())).all()


@pytest.mark.parametrize("nh,nkv,hd,window", [(32, 32, 64, 0), (32, 8, 48, 0), (32, 4, 16, 100), (32, 32, 64, 200),
                                              (32, 16, 32, 0), (32, 8, 128, 0), (8, 8, 96, 0), (40, 8, 64, 0), (16, 4, 64, 0),
                                              (16, 16, 64, 150)])
def test_tuned_prefill_long_portions(nh, nkv, hd, window):
    """Portions long enough, and heads enough, that a wave takes 64 tokens: one portion starts in the
    middle of its request and ends off every tile edge, the other is a whole short prompt."""
    from types import SimpleNamespace
    from glassbox_amd import ops
    q_lens, ctx_lens = [1101, 300], [1303, 300]
    k_pages, v_pages, tables, ks, vs = paged_setup(ctx_lens, nkv, hd, 16, seed=hd + nh, dtype=torch.bfloat16)
    ctx = BareContext(q_lens, ctx_lens, tables)
    n = sum(q_lens)
    q = (rnd(n, nh * hd, seed=12) * 0.7).bfloat16()
    scale = 1 / math.sqrt(hd)
    cache = SimpleNamespace(k_pages=to_dev(ops.pack_keys(k_pages)), v_pages=to_dev(v_pages), group=0)
    out = torch.zeros(n, nh * hd, device=DEV, dtype=torch.bfloat16)
    qd = to_dev(q)
    ops.attention_prefill(qd, out, ctx, cache, nh, scale, window)
    twin = torch.zeros_like(out)
    ops.attention_plain(qd, twin, ctx.positions, torch.tensor(ctx.tok_seq, dtype=torch.int32, device=DEV), ctx.tables[0],
                        cache.k_pages, cache.v_pages, nh, scale, window)
    close = (out.float() - twin.float()).abs() <= 2 ** -7 * (1 + twin.float().abs())
    bad = torch.nonzero(~close.all(dim=1)).flatten().tolist()
    assert not bad, f"rows {bad[:8]} (request, position) {[(ctx.tok_seq[i], ctx.pos_list[i]) for i in bad[:8]]}"
    # a sample of rows against the formula in float64: tile edges, the portion's ends, the second request
    rows = [0, 1, 31, 32, 63, 64, 127, 128, 255, 256, 257, 700, 1023, 1024, 1099, 1100, 1101, 1102, 1400]
    want = plain_attention_rows(q[rows], ks, vs, [ctx.tok_seq[i] for i in rows], [ctx.pos_list[i] for i in rows], nh,
                                scale, window)
    err = (out[rows].cpu().double() - want).abs().max().item()
    assert err < 2 ** -6, err


@pytest.mark.parametrize("nh,nkv,hd,window", [(8, 8, 64, 0), (16, 8, 32, 0), (8, 8, 128, 0), (24, 8, 48, 200)])
def test_tuned_decode_with_a_workgroup_per_request_and_kv_head(nh, nkv, hd, window):
    """Requests and kv heads enough that no context is split over workgroups: sixteen waves share one,
    and their results are combined within the workgroup."""
    from types import SimpleNamespace
    from glassbox_amd import ops
    g = torch.Generator().manual_seed(nh + hd)
    ctx_lens = [1, 2, 63, 64, 65, 255, 256, 257, 1023, 1024, 1025, 1500] + torch.randint(1, 1400, (24,), generator=g).tolist()
    assert ops.decode_chunk(len(ctx_lens), nkv, 1536) >= 1536          # one chunk takes it all
    k_pages, v_pages, tables, ks, vs = paged_setup(ctx_lens, nkv, hd, 16, seed=hd, dtype=torch.bfloat16)
    ctx = BareContext([1] * len(ctx_lens), ctx_lens, tables, max_context=1536)
    n = len(ctx_lens)
    q = (rnd(n, nh * hd, seed=13) * 0.7).bfloat16()
    scale = 1 / math.sqrt(hd)
    cache = SimpleNamespace(k_pages=to_dev(ops.pack_keys(k_pages)), v_pages=to_dev(v_pages), group=0)
    out = torch.zeros(n, nh * hd, device=DEV, dtype=torch.bfloat16)
    ops.attention_decode(to_dev(q), out, ctx, cache, nh, scale, window)
    want = plain_attention_rows(q, ks, vs, ctx.tok_seq, ctx.pos_list, nh, scale, window)
    err = (out.cpu().double() - want).abs().max(dim=1).values
    bad = torch.nonzero(err > 2 ** -6).flatten().tolist()
    assert not bad, f"requests {bad[:8]} with contexts {[ctx_lens[i] for i in bad[:8]]}: {err[bad[:8]]}"


@pytest.mark.parametrize("nh,nkv,hd,lens,bucket", [
    # one workgroup a context: its tiles of 64 keys in runs of up to five a wave, and in turns beyond 16 x 5 tiles
    (32, 32, 64, [1, 64, 65, 1024, 1025, 5119, 5120, 5121, 5184, 6143], 6144), (64, 32, 32, [5121, 320, 321, 5, 5056, 7000, 1, 6400], 7168),
    # up to 512 keys: one workgroup of four waves, also for one request
    (9, 3, 64, [1], 512), (8, 2, 128, [63, 64, 65, 257, 320, 321, 512], 512),
    # the sizes around which a whole context and chunks of it change over
    (10, 5, 64, [1000] * 16, 1024), (10, 5, 64, [999] * 15, 1024), (8, 8, 128, [2000] * 24, 2048), (8, 8, 128, [2000] * 23, 2048)])
def test_tuned_decode_whatever_a_workgroup_and_a_wave_take(nh, nkv, hd, lens, bucket):
    """Every way in which a context is dealt to workgroups and waves, against the plain kernel.  The values of each tile of 64 keys
    carry a mark in a dimension of the tile's, as much the larger as the tile has fewer keys: a mean over thousands of keys
    hardly shows which of them it left out, a mark that is not there does (512 / keys of some 0.8: 0.06 at 7,000, where the bound
    is 0.01)."""
    from types import SimpleNamespace
    from glassbox_amd import ops
    k_pages, v_pages, tables, ks, vs = paged_setup(lens, nkv, hd, 16, seed=hd + nkv, dtype=torch.bfloat16)
    for i, length in enumerate(lens):
        for at in range(0, length, 64):
            keys = min(64, length - at)
            for p in range(at, at + keys):
                v_pages[tables[i, p // 16], :, at // 64 % hd, p % 16] += 8 * 64 / keys
    ctx = BareContext([1] * len(lens), lens, tables, max_context=bucket)
    q = to_dev((rnd(len(lens), nh * hd, seed=13) * 0.7).bfloat16())
    cache = SimpleNamespace(k_pages=to_dev(ops.pack_keys(k_pages)), v_pages=to_dev(v_pages), group=0)
    out, twin = (torch.zeros(len(lens), nh * hd, device=DEV, dtype=torch.bfloat16) for _ in range(2))
    ops.attention_decode(q, out, ctx, cache, nh, 1 / math.sqrt(hd), 0)
    ops.attention_plain(q, twin, ctx.positions, torch.arange(len(lens), dtype=torch.int32, device=DEV), ctx.tables[0], cache.k_pages,
                        cache.v_pages, nh, 1 / math.sqrt(hd), 0)
    # softmax weights in bfloat16 (2^-9 of each value's share) and a bfloat16 result on either side
    assert ((out.float() - twin.float()).abs() <= 2 ** -7 * (1 + twin.float().abs())).all()


@pytest.mark.parametrize("nkv,G,hd,n,length,bucket,window,keep", [
    # a whole context a workgroup: more tiles a wave than a run holds, sixteen and four waves; runs; a window; kept first keys
    (32, 1, 64, 8, 5500, 6144, 0, 0), (8, 4, 128, 24, 1500, 2048, 0, 0), (32, 1, 64, 8, 4000, 4096, 0, 0),
    (32, 1, 64, 8, 3001, 3072, 1024, 0), (32, 1, 64, 8, 3001, 3072, 1024, 64), (8, 4, 128, 24, 1999, 2048, 300, 70),
    # chunks of a context
    (4, 2, 64, 3, 9000, 9216, 0, 0)])
def test_tuned_decode_gives_a_request_the_same_bits_in_every_row_and_head(nkv, G, hd, n, length, bucket, window, keep):
    """One request in every row of a step, its keys, values and queries alike in every head: the order in which a context is
    summed depends on sizes alone, so all heads of all rows are the same to the bit."""
    from types import SimpleNamespace
    from glassbox_amd import ops
    k_pages, v_pages, tables, _, _ = paged_setup([length], 1, hd, 16, seed=hd + nkv, dtype=torch.bfloat16)
    k_pages, v_pages = (t.expand(-1, nkv, -1, -1).contiguous() for t in (k_pages, v_pages))
    ctx = BareContext([1] * n, [length] * n, tables.expand(n, -1), max_context=bucket)
    q = to_dev((rnd(1, hd, seed=13) * 0.7).bfloat16().expand(n, nkv * G, hd).reshape(n, -1))
    cache = SimpleNamespace(k_pages=to_dev(ops.pack_keys(k_pages)), v_pages=to_dev(v_pages), group=0)
    out = torch.zeros(n, nkv * G * hd, device=DEV, dtype=torch.float32)
    ops.attention_decode(q, out, ctx, cache, nkv * G, 1 / math.sqrt(hd), window, keep)
    heads = out.view(n * nkv * G, hd)
    assert bool(heads[0].any()) and torch.equal(heads, heads[:1].expand_as(heads))


@pytest.mark.parametrize("nh,nkv,hd,lens,bucket,window", [
    # eight waves: a tile each or none, more tiles than waves in runs and beyond; the most workgroups, and one more; and where a bucket of
    # 512 or a window of up to 256 keys leaves them to four (the last workgroups that eight take, and more)
    (32, 32, 64, [500, 449, 64, 65, 510, 320, 17, 257], 510, 0), (15, 5, 16, [511], 511, 300), (15, 5, 16, [400, 511], 511, 256), (15, 5, 16, [400, 511], 511, 257),
    (12, 4, 64, [512, 30, 250, 320], 512, 0), (12, 4, 64, [512, 30, 250, 320, 1], 512, 0), (8, 4, 128, [300, 512] * 8, 512, 0), (8, 4, 128, [300, 512] * 8 + [9], 512, 0),
    (9, 3, 64, [257, 1, 300], 300, 0), (32, 32, 64, [512, 449, 64, 65, 500, 320, 17, 511], 512, 0), (15, 5, 16, [511], 512, 100),
    (32, 8, 128, [700] * 19 + [1, 129], 768, 0), (16, 8, 96, [2048, 1999] * 12, 2048, 0), (8, 4, 128, [1900] * 64, 2048, 300),
    (8, 4, 128, [300] * 65, 512, 0)])
def test_tuned_decode_of_whole_contexts_where_workgroups_are_few(nh, nkv, hd, lens, bucket, window):
    """Against the plain kernel, which sums a context a chunk of 256 keys after the other."""
    from types import SimpleNamespace
    from glassbox_amd import ops
    n = len(lens)
    assert ops.decode_chunk(n, nkv, bucket, hd) >= bucket
    k_pages, v_pages, tables, _, _ = paged_setup(lens, nkv, hd, 16, seed=hd + n, dtype=torch.bfloat16)
    q = to_dev((rnd(n, nh * hd, seed=6) * 0.7).bfloat16())
    ctx = BareContext([1] * n, lens, tables, max_context=bucket)
    cache = SimpleNamespace(k_pages=to_dev(ops.pack_keys(k_pages)), v_pages=to_dev(v_pages), group=0)
    out, twin = (torch.zeros(n, nh * hd, device=DEV, dtype=torch.bfloat16) for _ in range(2))
    ops.attention_decode(q, out, ctx, cache, nh, 1 / math.sqrt(hd), window)
    ops.attention_plain(q, twin, ctx.positions, torch.arange(n, dtype=torch.int32, device=DEV), ctx.tables[0], cache.k_pages,
                        cache.v_pages, nh, 1 / math.sqrt(hd), window)
    assert ((out.float() - twin.float()).abs() <= 2 ** -7 * (1 + twin.float().abs())).all()


def test_tuned_decode_finds_one_far_key_in_every_chunk_position():
    """One key is made to stand out: first and last slot of a page, chunk edges, the last position."""
    from types import SimpleNamespace
    from glassbox_amd import ops
    nh, nkv, hd, page, ctxlen = 4, 2, 64, 16, 1500
    k_pages, v_pages, tables, ks, vs = paged_setup([ctxlen], nkv, hd, page, seed=1, dtype=torch.bfloat16)
    q = rnd(1, nh * hd, seed=2).float().reshape(nh, hd)
    q[1::2] = q[0::2]
    q = q.reshape(1, nh * hd).bfloat16()
    for target in (0, 15, 16, 63, 64, 255, 256, 257, 511, 512, 1023, 1024, 1279, 1280, 1498, 1499):
        kp = k_pages.clone()
        for kvh in range(nkv):
            kp[tables[0, target // page], kvh, target % page, :] = (q[0].float().reshape(nh, hd)[2 * kvh] * 40).bfloat16()
        for max_context in (1500, 4096):                       # one and several chunks per workgroup
            ctx = BareContext([1], [ctxlen], tables, max_context=max_context)
            out = torch.zeros(1, nh * hd, device=DEV, dtype=torch.bfloat16)
            cache = SimpleNamespace(k_pages=to_dev(ops.pack_keys(kp)), v_pages=to_dev(v_pages), group=0)
            ops.attention_decode(to_dev(q), out, ctx, cache, nh, 1 / math.sqrt(hd), 0)
            want = vs[0][target].float().repeat_interleave(2, 0).reshape(-1)
            assert (out.cpu().float()[0] - want).abs().max().item() < 2e-2, f"key at {target} was not found"


@pytest.mark.parametrize("page,ctxlen", [(1200016, 1200216), (48, 70000), (65552, 131204)])
def test_tuned_decode_finds_a_key_in_pages_of_any_size(page, ctxlen):
    """Page numbers come by a multiplication: pages that are no power of two, up to ones of more than a million keys.  All keys are zeros but
    one: at the ends of pages, of the context, and of a chunk."""
    from types import SimpleNamespace
    from glassbox_amd import ops
    nh, nkv, hd = 2, 1, 16
    n_pages = -(-ctxlen // page)
    chunk = ops.decode_chunk(1, nkv, ctxlen, hd)
    values = rnd(ctxlen, hd, seed=3).bfloat16()
    v_pages = torch.zeros(n_pages, page, hd, dtype=torch.bfloat16)
    v_pages.view(-1, hd)[:ctxlen] = values
    tables = torch.arange(n_pages, dtype=torch.int32).flip(0)[None]          # the last page first
    v_pages = to_dev(v_pages[tables[0].long()].transpose(1, 2)[:, None].contiguous())
    q = rnd(1, nh * hd, seed=2).bfloat16()
    q[0, hd:] = q[0, :hd]
    for target in (0, page - 1, page, ctxlen - 1, chunk - 1, chunk):
        k_pages = torch.zeros(n_pages, nkv, page, hd, dtype=torch.bfloat16)
        k_pages[tables[0, target // page], 0, target % page] = q[0, :hd] * 40
        cache = SimpleNamespace(k_pages=to_dev(ops.pack_keys(k_pages)), v_pages=v_pages, group=0)
        out = torch.zeros(1, nh * hd, device=DEV, dtype=torch.bfloat16)
        ops.attention_decode(to_dev(q), out, BareContext([1], [ctxlen], tables, max_context=ctxlen), cache, nh, 1 / math.sqrt(hd), 0)
        # (its weight is e^(10 |q|^2), of the others together ctxlen)
        assert (out.cpu().float().view(nh, hd) - values[target].float()).abs().max().item() < 2e-2, f"key at {target} was not found"


@pytest.mark.parametrize("layout", ["a column turned", "one row for all", "rows over each other", "the end of a wider table", "the middle of one"])
def test_tuned_decode_takes_block_tables_of_any_row_stride(layout):
    """A row's first entries are asked for before the position is known, wherever the rows lie: the bits of tables of their own."""
    from types import SimpleNamespace
    from glassbox_amd import ops
    nh, nkv, hd, n = 6, 2, 64, 1 if layout == "a column turned" else 3
    k_pages, v_pages, tables, _, _ = paged_setup([300], nkv, hd, 16, seed=8, dtype=torch.bfloat16)
    width = tables.shape[1]
    rows = tables.expand(n, -1).contiguous()
    if layout == "a column turned":
        view = to_dev(tables[0][:, None].contiguous()).t()
    elif layout == "one row for all":
        view = to_dev(tables).expand(n, -1)
    elif layout == "rows over each other":
        view = torch.as_strided(to_dev(torch.cat([tables[0], tables[0][:4]])), (n, width), (2, 1))
        rows = view.cpu().contiguous()
    else:
        below, at = (0, 9) if layout == "the end of a wider table" else (1, 4)
        wide = torch.full((n + below, width + 9), -1, dtype=torch.int32)
        wide[:n, at:at + width] = rows
        view = to_dev(wide)[:n, at:at + width]
    lens = [300, 17, 290][:n]
    q = to_dev((rnd(n, nh * hd, seed=6) * 0.7).bfloat16())
    cache = SimpleNamespace(k_pages=to_dev(ops.pack_keys(k_pages)), v_pages=to_dev(v_pages), group=0)
    outs = []
    for t in (to_dev(rows), view):
        ctx = BareContext([1] * n, lens, rows, max_context=300)
        ctx.tables = [t]
        out = torch.zeros(n, nh * hd, device=DEV, dtype=torch.bfloat16)
        ops.attention_decode(q, out, ctx, cache, nh, 1 / math.sqrt(hd), 0)
        outs.append(out.cpu())
    assert view.stride() != to_dev(rows).stride() and torch.equal(*outs)


def test_tuned_decode_over_tens_of_thousands_of_keys():
    """Contexts of 40,000 and 33,333 keys beside one of 5: some hundred and sixty chunks a request for the second
    pass to merge, block tables of 2,500 pages.  Against the plain kernel on random keys, and with one key made to
    stand out near the start, in the middle and at the end."""
    from types import SimpleNamespace
    from glassbox_amd import ops
    nh, nkv, hd, page = 4, 2, 64, 16
    ctx_lens = [40000, 33333, 5]
    k_pages, v_pages, tables, ks, vs = paged_setup(ctx_lens, nkv, hd, page, seed=5, dtype=torch.bfloat16)
    q = (rnd(3, nh * hd, seed=6) * 0.7).bfloat16()
    ctx = BareContext([1, 1, 1], ctx_lens, tables, max_context=40960)
    assert -(-40960 // ops.decode_chunk(3, nkv, 40960)) > 100
    cache = SimpleNamespace(k_pages=to_dev(ops.pack_keys(k_pages)), v_pages=to_dev(v_pages), group=0)
    out, twin = (torch.zeros(3, nh * hd, device=DEV, dtype=torch.bfloat16) for _ in range(2))
    ops.attention_decode(to_dev(q), out, ctx, cache, nh, 1 / math.sqrt(hd), 0)
    ops.attention_plain(to_dev(q), twin, ctx.positions, torch.tensor([0, 1, 2], dtype=torch.int32, device=DEV), ctx.tables[0],
                        cache.k_pages, cache.v_pages, nh, 1 / math.sqrt(hd), 0)
    assert ((out.float() - twin.float()).abs() <= 2 ** -7 * (1 + twin.float().abs())).all()
    qq = q.float().reshape(3, nh, hd)
    qq[:, 1::2] = qq[:, 0::2]
    qq = qq.reshape(3, nh * hd).bfloat16()
    for target in (3, 20479, 20480, 39999):
        kp = k_pages.clone()
        for kvh in range(nkv):
            kp[tables[0, target // page], kvh, target % page, :] = (qq[0].float().reshape(nh, hd)[2 * kvh] * 40).bfloat16()
        cache = SimpleNamespace(k_pages=to_dev(ops.pack_keys(kp)), v_pages=to_dev(v_pages), group=0)
        ops.attention_decode(to_dev(qq), out, ctx, cache, nh, 1 / math.sqrt(hd), 0)
        want = vs[0][target].float().repeat_interleave(2, 0).reshape(-1)
        assert (out.cpu().float()[0] - want).abs().max().item() < 2e-2, f"key at {target} of 40,000 was not found"


@pytest.mark.parametrize("nh,nkv,hd,window", [(8, 2, 64, 0), (4, 4, 128, 0), (6, 3, 32, 700), (8, 8, 96, 0)])
def test_tuned_prefill_short_portions_over_long_contexts(nh, nkv, hd, window):
    """Few pairs of blocks and long contexts: several workgroups share a pair's keys and a second pass adds their
    sums.  Two short portions at the ends of long requests, beside a request of a single token."""
    from types import SimpleNamespace
    from glassbox_amd import ops
    q_lens, ctx_lens = [1, 100, 37], [400, 2150, 1301]
    k_pages, v_pages, tables, ks, vs = paged_setup(ctx_lens, nkv, hd, 16, seed=hd + nh, dtype=torch.bfloat16)
    ctx = BareContext(q_lens, ctx_lens, tables)
    lib = ops._lib("attention_bf16")
    assert lib.gb_attention_prefill_parts(max(q_lens), max(ctx_lens), nh, 2, hd) > 1
    n = sum(q_lens)
    q = (rnd(n, nh * hd, seed=14) * 0.7).bfloat16()
    scale = 1 / math.sqrt(hd)
    cache = SimpleNamespace(k_pages=to_dev(ops.pack_keys(k_pages)), v_pages=to_dev(v_pages), group=0)
    out = torch.zeros(n, nh * hd, device=DEV, dtype=torch.bfloat16)
    qd = to_dev(q)
    ops.attention_decode(qd, out, ctx, cache, nh, scale, window)
    ops.attention_prefill(qd, out, ctx, cache, nh, scale, window)
    twin = torch.zeros_like(out)
    ops.attention_plain(qd, twin, ctx.positions, torch.tensor(ctx.tok_seq, dtype=torch.int32, device=DEV), ctx.tables[0],
                        cache.k_pages, cache.v_pages, nh, scale, window)
    close = (out.float() - twin.float()).abs() <= 2 ** -7 * (1 + twin.float().abs())
    bad = torch.nonzero(~close.all(dim=1)).flatten().tolist()
    assert not bad, f"rows {bad[:8]} (request, position) {[(ctx.tok_seq[i], ctx.pos_list[i]) for i in bad[:8]]}"
    want = plain_attention_rows(q, ks, vs, ctx.tok_seq, ctx.pos_list, nh, scale, window)
    assert (out.cpu().double() - want).abs().max().item() < 2 ** -6
    again = torch.zeros_like(out)
    ops.attention_decode(qd, again, ctx, cache, nh, scale, window)
    ops.attention_prefill(qd, again, ctx, cache, nh, scale, window)
    assert torch.equal(out, again)


@pytest.mark.parametrize("nh,nkv,hd,window,keep,chunk", [(8, 2, 64, 700, 70, 0), (8, 8, 128, 300, 0, 0), (4, 4, 64, 0, 0, 1024)])
def test_tuned_prefill_behind_histories_that_windows_and_runs_leave_out(nh, nkv, hd, window, keep, chunk):
    """Short portions behind long contexts of which their tokens see little: the launch is shaped by what they see, the same
    results as the plain kernel's, and no workspace of a longer context's size is asked for."""
    from types import SimpleNamespace
    from glassbox_amd import ops
    q_lens, ctx_lens = [100, 37], [5150, 3301]
    k_pages, v_pages, tables, _, _ = paged_setup(ctx_lens, nkv, hd, 16, seed=hd + nh, dtype=torch.bfloat16)
    ctx = BareContext(q_lens, ctx_lens, tables)
    q = to_dev((rnd(sum(q_lens), nh * hd, seed=14) * 0.7).bfloat16())
    cache = SimpleNamespace(k_pages=to_dev(ops.pack_keys(k_pages)), v_pages=to_dev(v_pages), group=0)
    out, twin = torch.zeros_like(q), torch.zeros_like(q)
    ops.attention_prefill(q, out, ctx, cache, nh, 1 / math.sqrt(hd), window, keep, chunk)
    parts = ops._prefill_parts(max(q_lens), (window + keep or chunk) + max(q_lens), nh, 2, hd)
    assert parts < ops._prefill_parts(max(q_lens), max(ctx_lens), nh, 2, hd)
    assert [k[1][0] for k in ctx._bufs] == ([parts * sum(q_lens) * nh * (hd + 2)] if parts > 1 else [])
    ops.attention_plain(q, twin, ctx.positions, torch.tensor(ctx.tok_seq, dtype=torch.int32, device=DEV), ctx.tables[0],
                        cache.k_pages, cache.v_pages, nh, 1 / math.sqrt(hd), window, keep_first=keep, chunk=chunk)
    assert ((out.float() - twin.float()).abs() <= 2 ** -7 * (1 + twin.float().abs())).all()


@pytest.mark.parametrize("shape,nh,nkv,hd,q_lens,history,window,keep,chunk", [
    # one tile of keys; a request of one block beside one of two; a block whose last token is its first
    (211, 6, 2, 64, [33, 2, 64], 0, 0, 0, 0), (211, 8, 8, 128, [64, 31], 0, 0, 0, 0),
    # two waves a block: three tiles (the last one a wave's alone); a window that leaves out tiles of the later blocks, kept keys
    (221, 15, 5, 64, [65, 190], 0, 0, 0, 0), (221, 32, 32, 64, [1025], 0, 300, 70, 0), (221, 8, 1, 128, [257], 40, 0, 0, 0),
    # four waves a block: five tiles, and one tile for some tokens; runs of positions; a group of three heads over two blocks
    (241, 9, 3, 64, [300, 17], 0, 0, 0, 0), (241, 8, 8, 64, [700], 33, 0, 0, 256), (241, 9, 3, 64, [129], 1300, 200, 20, 0),
    # four blocks a workgroup, of one head and of several; a last workgroup of one block
    (411, 32, 32, 64, [161] * 8, 0, 0, 0, 0), (411, 32, 4, 128, [300, 295, 225, 33], 0, 0, 0, 0), (411, 64, 16, 64, [545, 3290], 0, 0, 0, 0),
    (421, 40, 8, 64, [2081], 0, 0, 0, 0), (421, 32, 32, 128, [1000], 0, 150, 64, 0),
    # several workgroups a block's keys: parts of unequal tiles, all eight, and tokens that see none of a part's
    (225, 32, 32, 64, [131], 1500, 0, 0, 0), (228, 4, 2, 64, [40, 3], 2700, 0, 0, 0), (224, 8, 2, 128, [100, 37], 2000, 0, 0, 0),
    (223, 6, 2, 64, [90], 3000, 1000, 30, 0)])
@pytest.mark.parametrize("page", [16, 32, 128])
def test_tuned_prefill_of_every_shape(shape, nh, nkv, hd, q_lens, history, window, keep, chunk, page):
    """The kernel whose waves share tiles of keys, in each of its workgroups' shapes (blocks a workgroup, waves a block,
    workgroups a block's keys), against the plain kernel; result rows wider than the heads are left alone."""
    from types import SimpleNamespace
    from glassbox_amd import ops
    seen = max(q_lens) + (min(history, window + keep) if window else history)
    assert ops._lib("attention_bf16").gb_attention_prefill_shape(max(q_lens), seen, nh, len(q_lens), hd) == shape
    ctx_lens = [history + n for n in q_lens]
    k_pages, v_pages, tables, _, _ = paged_setup(ctx_lens, nkv, hd, page, seed=hd + nh, dtype=torch.bfloat16)
    ctx = BareContext(q_lens, ctx_lens, tables)
    q = to_dev((rnd(sum(q_lens), nh * hd, seed=14) * 0.7).bfloat16())
    cache = SimpleNamespace(k_pages=to_dev(ops.pack_keys(k_pages)), v_pages=to_dev(v_pages), group=0)
    wide = torch.full((sum(q_lens), nh * hd + 8), 7.0, device=DEV, dtype=torch.bfloat16)
    sinks = to_dev(rnd(nh, seed=5).float()) if chunk or window else None
    twin = torch.zeros_like(q)
    ops.attention_prefill(q, wide[:, :nh * hd], ctx, cache, nh, 1 / math.sqrt(hd), window, keep, chunk, sinks=sinks)
    ops.attention_plain(q, twin, ctx.positions, torch.tensor(ctx.tok_seq, dtype=torch.int32, device=DEV), ctx.tables[0],
                        cache.k_pages, cache.v_pages, nh, 1 / math.sqrt(hd), window, keep_first=keep, chunk=chunk, sinks=sinks)
    # softmax weights in bfloat16 (2^-9 of each value's share) and a bfloat16 result on either side
    close = (wide[:, :nh * hd].float() - twin.float()).abs() <= 2 ** -7 * (1 + twin.float().abs())
    bad = torch.nonzero(~close.all(dim=1)).flatten().tolist()
    assert not bad, f"rows {bad[:8]} (request, position) {[(ctx.tok_seq[i], ctx.pos_list[i]) for i in bad[:8]]}"
    assert bool((wide[:, nh * hd:] == 7.0).all())


@pytest.mark.parametrize("nh,nkv,hd", [(4, 2, 16), (6, 2, 32), (2, 1, 48), (6, 3, 64), (4, 4, 80), (3, 1, 96), (2, 2, 112), (4, 2, 128)])
@pytest.mark.parametrize("window,keep,q_lens,history", [(44, 200, [572, 14], 0), (44, 200, [85, 300], 53), (20, 97, [400], 0), (100, 65, [33, 700], 0),
                                                        (16, 130, [333], 7), (300, 500, [900], 0), (44, 200, [300], 1605)])
@pytest.mark.parametrize("softcap,wide", [(0.0, False), (20.0, False), (0.0, True)])
def test_tuned_prefill_with_more_kept_first_keys_than_a_tile_holds(nh, nkv, hd, window, keep, q_lens, history, softcap, wide):
    """A prompt's first tokens see few of the kept keys, its last ones all of them, beside a window that begins far behind: every
    kernel and way of sharing the keys, against the plain kernel."""
    from types import SimpleNamespace
    from glassbox_amd import ops
    ctx_lens = [history + n for n in q_lens]
    k_pages, v_pages, tables, _, _ = paged_setup(ctx_lens, nkv, hd, 16, seed=hd + nh, dtype=torch.bfloat16)
    ctx = BareContext(q_lens, ctx_lens, tables)
    q = to_dev((rnd(sum(q_lens), nh * hd, seed=14) * 0.7).bfloat16())
    cache = SimpleNamespace(k_pages=to_dev(ops.pack_keys(k_pages)), v_pages=to_dev(v_pages), group=0)
    out, twin = (torch.zeros(q.shape, device=DEV, dtype=torch.float32 if wide else torch.bfloat16) for _ in range(2))
    twin = torch.zeros_like(q)
    ops.attention_prefill(q, out, ctx, cache, nh, 1 / math.sqrt(hd), window, keep, softcap=softcap)
    ops.attention_plain(q, twin, ctx.positions, torch.tensor(ctx.tok_seq, dtype=torch.int32, device=DEV), ctx.tables[0],
                        cache.k_pages, cache.v_pages, nh, 1 / math.sqrt(hd), window, keep_first=keep, softcap=softcap)
    # softmax weights in bfloat16 (2^-9 of each value's share) and a bfloat16 result on either side
    close = (out.float() - twin.float()).abs() <= 2 ** -7 * (1 + twin.float().abs())
    bad = torch.nonzero(~close.all(dim=1)).flatten().tolist()
    assert not bad, f"{len(bad)} rows, {bad[:8]} (request, position) {[(ctx.tok_seq[i], ctx.pos_list[i]) for i in bad[:8]]}"


@pytest.mark.parametrize("shape,nh,nkv,hd,q_lens,history", [
    (228, 4, 2, 64, [3, 40], [0, 2700]), (227, 4, 2, 64, [40, 2, 33], [2300, 0, 70]), (226, 6, 3, 64, [17, 64], [1, 2100]),
    (228, 4, 1, 128, [3, 40], [0, 4200]), (225, 4, 4, 128, [60, 2], [2700, 130])])
@pytest.mark.parametrize("page", [16, 64])
def test_tuned_prefill_of_short_requests_beside_long_ones(shape, nh, nkv, hd, q_lens, history, page):
    """Requests with fewer tiles of keys than the workgroups that the longest one's are spread over: some of theirs have no tile,
    and hand over nothing."""
    from types import SimpleNamespace
    from glassbox_amd import ops
    ctx_lens = [h + n for h, n in zip(history, q_lens)]
    assert ops._lib("attention_bf16").gb_attention_prefill_shape(max(q_lens), max(ctx_lens), nh, len(q_lens), hd) == shape
    k_pages, v_pages, tables, _, _ = paged_setup(ctx_lens, nkv, hd, page, seed=hd + nh, dtype=torch.bfloat16)
    ctx = BareContext(q_lens, ctx_lens, tables)
    q = to_dev((rnd(sum(q_lens), nh * hd, seed=14) * 0.7).bfloat16())
    cache = SimpleNamespace(k_pages=to_dev(ops.pack_keys(k_pages)), v_pages=to_dev(v_pages), group=0)
    out, twin = torch.zeros_like(q), torch.zeros_like(q)
    ops.attention_prefill(q, out, ctx, cache, nh, 1 / math.sqrt(hd), 0)
    ops.attention_plain(q, twin, ctx.positions, torch.tensor(ctx.tok_seq, dtype=torch.int32, device=DEV), ctx.tables[0],
                        cache.k_pages, cache.v_pages, nh, 1 / math.sqrt(hd), 0)
    # softmax weights in bfloat16 (2^-9 of each value's share) and a bfloat16 result on either side
    assert ((out.float() - twin.float()).abs() <= 2 ** -7 * (1 + twin.float().abs())).all()


@pytest.mark.parametrize("shape,nh,nkv,hd,q_lens,history", [
    # few tiles; from nine or eleven on several workgroups a block; many requests; beyond a workgroup a unit; three parts of long ones
    (221, 8, 2, 128, [31, 2], 480), (223, 8, 2, 128, [31, 2], 500), (221, 33, 33, 128, [31, 2], 600), (223, 8, 2, 128, [31, 2], 640), (224, 9, 3, 128, [17], 860), (221, 32, 8, 128, [5] * 17, 700),
    (211, 32, 32, 128, [3, 32, 17] * 3, 150), (223, 43, 43, 128, [20, 9, 31], 3050), (222, 40, 8, 128, [32, 3] * 2, 1100),
    (221, 32, 32, 64, [3, 32, 17] * 3, 300), (221, 15, 5, 64, [31, 2] * 13, 250), (241, 15, 5, 64, [31, 2] * 12, 250)])
def test_tuned_prefill_of_portions_of_one_block(shape, nh, nkv, hd, q_lens, history):
    """Portions of up to 32 tokens, whose workgroups hold query heads of a kv head side by side: every way of spreading them, and
    blocks with columns without a token."""
    from types import SimpleNamespace
    from glassbox_amd import ops
    ctx_lens = [history + n for n in q_lens]
    lib = ops._lib("attention_bf16")
    assert lib.gb_attention_prefill_shape_of(max(q_lens), max(ctx_lens), nh, nkv, len(q_lens), hd) == shape
    assert ops._prefill_parts(max(q_lens), max(ctx_lens), nh, len(q_lens), hd) >= shape % 10
    k_pages, v_pages, tables, _, _ = paged_setup(ctx_lens, nkv, hd, 16, seed=hd + nh, dtype=torch.bfloat16)
    ctx = BareContext(q_lens, ctx_lens, tables)
    q = to_dev((rnd(sum(q_lens), nh * hd, seed=14) * 0.7).bfloat16())
    cache = SimpleNamespace(k_pages=to_dev(ops.pack_keys(k_pages)), v_pages=to_dev(v_pages), group=0)
    for window, keep, chunk in ((0, 0, 0), (history - 60, 20, 0), (0, 0, history - 33)):
        out, twin = torch.zeros_like(q), torch.zeros_like(q)
        ops.attention_prefill(q, out, ctx, cache, nh, 1 / math.sqrt(hd), window, keep, chunk)
        ops.attention_plain(q, twin, ctx.positions, torch.tensor(ctx.tok_seq, dtype=torch.int32, device=DEV), ctx.tables[0],
                            cache.k_pages, cache.v_pages, nh, 1 / math.sqrt(hd), window, keep_first=keep, chunk=chunk)
        # softmax weights in bfloat16 (2^-9 of each value's share) and a bfloat16 result on either side
        assert ((out.float() - twin.float()).abs() <= 2 ** -7 * (1 + twin.float().abs())).all()


@pytest.mark.parametrize("group", [1, 2, 3, 4, 6, 12])
@pytest.mark.parametrize("hd", [64, 128])
def test_the_workspace_of_a_portion_suffices_for_any_number_of_kv_heads(group, hd):
    from glassbox_amd import ops
    lib = ops._lib("attention_bf16")
    for nkv in (1, 2, 5, 8, 11, 32):
        for n in (1, 2, 3, 5, 8, 17, 40):
            for q_len in (3, 32, 33, 200):
                for context in (q_len, 600, 710, 1100, 3100, 8000):
                    shape = lib.gb_attention_prefill_shape_of(q_len, context, nkv * group, nkv, n, hd)
                    assert 1 <= shape % 10 <= ops._prefill_parts(q_len, context, nkv * group, n, hd)


@pytest.mark.parametrize("nh,ctxlen,qlen", [(2, 200, 90), (64, 1200, 1090)])   # 32 and 64 tokens a wave
def test_tuned_prefill_sees_exactly_the_causal_keys(nh, ctxlen, qlen):
    """A portion in the middle of a request (it starts at position 110): token t must find a marked
    key at its own position and must not see the one after it."""
    from types import SimpleNamespace
    from glassbox_amd import ops
    nkv, hd, page = 2, 64, 16
    k_pages, v_pages, tables, ks, vs = paged_setup([ctxlen], nkv, hd, page, seed=3, dtype=torch.bfloat16)
    ctx = BareContext([qlen], [ctxlen], tables)
    # every key lies along one axis with a length that grows with its position, through consecutive
    # bfloat16 numbers from 16.0 on (so that rounding cannot reorder them): the newest visible key wins
    lengths = (torch.arange(ctxlen, dtype=torch.int32) + 0x4180).to(torch.int16).view(torch.bfloat16)
    axis = torch.zeros(hd)
    axis[5] = 1.0
    kp = k_pages.clone()
    for p in range(ctxlen):
        kp[tables[0, p // page], :, p % page, :] = (axis * lengths[p].float()).bfloat16()
    q = (axis * 768).repeat(qlen, nh).bfloat16()             # neighbours differ by 12 and more in score
    out = torch.zeros(qlen, nh * hd, device=DEV, dtype=torch.bfloat16)
    cache = SimpleNamespace(k_pages=to_dev(ops.pack_keys(kp)), v_pages=to_dev(v_pages), group=0)
    ops.attention_prefill(to_dev(q), out, ctx, cache, nh, 1 / math.sqrt(hd), 0)
    got = out.cpu().float().reshape(qlen, nkv, nh // nkv, hd)
    want = vs[0][110:110 + qlen].float()[:, :, None, :]      # not the value of the position after it
    worst = (got - want).abs().amax(dim=(1, 2, 3))
    assert worst.max().item() < 3e-2, f"token {int(worst.argmax())} of the portion"


def test_copy_rows():
    from glassbox_amd import ops
    base = rnd(6, 3, 10, seed=1).to(DEV)
    want = base.clone()
    want[4], want[0] = want[1].clone(), want[5].clone()
    ops.copy_rows(base, torch.tensor([1, 5], dtype=torch.int32, device=DEV), torch.tensor([4, 0], dtype=torch.int32, device=DEV))
    assert torch.equal(base, want)

