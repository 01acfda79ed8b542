"""Each kernel alone against a plain reference of the same operation, at sizes other than the engine's."""
import math

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _rel(got, want):
    want = want.double()
    return float((got.double() - want).abs().max() / want.abs().max().clamp_min(1e-30))


# --- matrix products -----------------------------------------------------------------------------
GEMM_SHAPES = [(1, 48, 64), (7, 300, 96), (8, 3584, 512), (16, 200, 128), (17, 331, 80), (33, 1000, 264),
               (64, 520, 1024), (65, 130, 72), (128, 128, 64), (100, 9000, 72), (200, 257, 136), (515, 384, 200),
               (2050, 4100, 136)]   # the last ones take each tiling of the tiled kernel


@pytest.mark.parametrize("m,n,k", GEMM_SHAPES)
@pytest.mark.parametrize("out_dtype", [torch.float32, torch.bfloat16])
def test_gemm_bf16_against_float64(m, n, k, out_dtype):
    from vipera_rs_amd.ops import kernels
    g = torch.Generator().manual_seed(m * 1000 + n + k)
    a = torch.randn(m, k, generator=g).to(torch.bfloat16).to(DEV)
    w = torch.randn(n, k, generator=g).to(torch.bfloat16).to(DEV)
    bias = torch.randn(n, generator=g).to(DEV)
    want = a.double() @ w.double().T + bias.double()
    out = torch.empty(m, n, dtype=out_dtype, device=DEV)
    kernels.gemm_bf16(a, w, bias, out)
    tol = 1e-5 if out_dtype == torch.float32 else 6e-3
    assert _rel(out, want) < tol
    if out_dtype == torch.float32:  # accumulation into a 32-bit residual, no bias
        base = torch.randn(m, n, generator=g).to(DEV)
        acc = base.clone()
        kernels.gemm_bf16(a, w, None, acc, accumulate=True)
        assert _rel(acc, base.double() + a.double() @ w.double().T) < 1e-5


@pytest.mark.parametrize("tiling", [0, 2, 3, 4, 9, 7, 8, 5])
@pytest.mark.parametrize("ranges", [1, 2, 8])
def test_gemm_bf16_every_tiling_of_the_tiled_kernel(tiling, ranges):
    """Each tiling of both tiled kernels, forced: tails in both directions, one to many K steps (an odd
    number too, so both LDS stages end a run), K split into ranges, and a K that the direct kernel passes on."""
    from vipera_rs_amd.ops import kernels
    shapes = [(257, 520, 1024), (129, 1028, 128), (300, 264, 64), (513, 300, 1600), (65, 2100, 4608), (200, 257, 136)]
    try:
        kernels.gemm_bf16_force_tiling(tiling, ranges)
        for m, n, k in shapes:
            g = torch.Generator().manual_seed(m + n + k)
            a = torch.randn(m, k, generator=g).to(torch.bfloat16).to(DEV)
            w = torch.randn(n, k, generator=g).to(torch.bfloat16).to(DEV)
            bias = torch.randn(n, generator=g).to(DEV)
            product = a.double() @ w.double().T
            for out_dtype, tol in ((torch.float32, 1e-5), (torch.bfloat16, 6e-3)):
                out = torch.full((m, n), 7.0, dtype=out_dtype, device=DEV)
                kernels.gemm_bf16(a, w, bias, out)
                assert _rel(out, product + bias.double()) < tol, (m, n, k, out_dtype)
            base = torch.randn(m, n, generator=g).to(DEV)
            acc = base.clone()
            kernels.gemm_bf16(a, w, None, acc, accumulate=True)
            assert _rel(acc, base.double() + product) < 1e-5, (m, n, k, "accumulate")
    finally:
        kernels.gemm_bf16_force_tiling(-1)


@pytest.mark.parametrize("tiling", [13, 14, 15])
@pytest.mark.parametrize("ranges", [1, 2, 3, 8])
def test_the_small_tilings_give_the_bits_of_the_large_one(tiling, ranges):
    """64x64 and 128x64 tiles with three and four LDS stages, K split over workgroups or its ranges added up in one:
    the same sums in the same order as the 128x128 tiles with as many ranges.  Tails in both directions, runs shorter
    than the stages, ranges that end in every stage and that K does not fill."""
    from vipera_rs_amd.ops import kernels
    from vipera_rs_amd.ops.linear import interleave_gate_up
    try:
        for m, n, k in [(129, 33, 64), (200, 96, 128), (257, 130, 192), (300, 264, 256), (150, 64, 1600), (513, 301, 1088), (140, 520, 4096)]:
            g = torch.Generator().manual_seed(m + n + k)
            a = torch.randn(m, k, generator=g).to(torch.bfloat16).to(DEV)
            w = torch.randn(n, k, generator=g).to(torch.bfloat16).to(DEV)
            bias, base = torch.randn(n, generator=g).to(DEV), torch.randn(m, n, generator=g).to(DEV)
            fused = interleave_gate_up(w[:n // 16 * 16], w[:n // 16 * 16].flip(0).contiguous())
            got = []
            for now in (9, tiling):
                kernels.gemm_bf16_force_tiling(now, ranges)
                outs = [torch.full((m, n), 7.0, device=DEV), torch.full((m, n), 7.0, dtype=torch.bfloat16, device=DEV), base.clone(),
                        torch.full((m, n // 16 * 16), 7.0, dtype=torch.bfloat16, device=DEV)]
                kernels.gemm_bf16(a, w, bias, outs[0])
                kernels.gemm_bf16(a, w, None, outs[1])
                kernels.gemm_bf16(a, w, None, outs[2], accumulate=True)
                kernels.gemm_bf16_gated(a, fused, outs[3])
                got.append(outs)
            assert all(torch.equal(x, y) for x, y in zip(*got)), (m, n, k)
            assert _rel(got[1][0], a.double() @ w.double().T + bias.double()) < 1e-5, (m, n, k)
    finally:
        kernels.gemm_bf16_force_tiling(-1)


@pytest.mark.parametrize("tiling", [16, 17, 18, 19, 20])
@pytest.mark.parametrize("ranges", [1, 3])
def test_the_tiles_of_whole_products_give_the_bits_of_the_128x128_ones(tiling, ranges):
    """192x64, 128x128, 192x128 and 192x192 tiles with two to four LDS stages: tails of a row and a column, runs shorter than
    the stages and runs that end in every stage, several rounds of tiles, plain, added to a residual and gated."""
    from vipera_rs_amd.ops import kernels
    from vipera_rs_amd.ops.linear import interleave_gate_up
    try:
        for m, n, k in [(129, 33, 64), (193, 65, 128), (385, 193, 192), (192, 192, 256), (191, 300, 320), (577, 129, 1088), (140, 520, 2048)]:
            g = torch.Generator().manual_seed(m + n + k)
            a = torch.randn(m, k, generator=g).to(torch.bfloat16).to(DEV)
            w = torch.randn(n, k, generator=g).to(torch.bfloat16).to(DEV)
            bias, base = torch.randn(n, generator=g).to(DEV), torch.randn(m, n, generator=g).to(DEV)
            fused = interleave_gate_up(w[:n // 16 * 16], w[:n // 16 * 16].flip(0).contiguous())
            got = []
            for now in (9, tiling):
                kernels.gemm_bf16_force_tiling(now, ranges)
                outs = [torch.full((m, n), 7.0, device=DEV), torch.full((m, n), 7.0, dtype=torch.bfloat16, device=DEV), base.clone(),
                        torch.full((m, n // 16 * 16), 7.0, dtype=torch.bfloat16, device=DEV)]
                kernels.gemm_bf16(a, w, bias, outs[0])
                kernels.gemm_bf16(a, w, None, outs[1])
                kernels.gemm_bf16(a, w, None, outs[2], accumulate=True)
                kernels.gemm_bf16_gated(a, fused, outs[3])
                got.append(outs)
            assert all(torch.equal(x, y) for x, y in zip(*got)), (m, n, k)
            assert _rel(got[1][0], a.double() @ w.double().T + bias.double()) < 1e-5, (m, n, k)
    finally:
        kernels.gemm_bf16_force_tiling(-1)


@pytest.mark.parametrize("tiling", [5, 6, 9])
def test_tiles_with_a_third_stage_of_the_weight_give_the_bits_of_the_others(tiling):
    """Runs of K shorter than the stages, as long, and ending in every pair of stages (64 to 640), whole and in ranges, with tails
    of a row and a column: the bits of the 256x128 tiles, whose operands have three stages each."""
    from vipera_rs_amd.ops import kernels
    g = torch.Generator().manual_seed(tiling)
    for m, n in ((257, 288), (300, 416)):
        for k in (64, 128, 192, 256, 320, 384, 640, 1152):
            a = torch.randn(m, k, generator=g).to(torch.bfloat16).to(DEV)
            w = torch.randn(n, k, generator=g).to(torch.bfloat16).to(DEV)
            for ranges in (1, 2):
                got = []
                try:
                    for one in (tiling, 7):
                        kernels.gemm_bf16_force_tiling(one, ranges)
                        outs = [torch.full((m, n), 7.0, device=DEV), torch.full((m, n // 2), 7.0, dtype=torch.bfloat16, device=DEV)]
                        kernels.gemm_bf16(a, w, None, outs[0])
                        kernels.gemm_bf16_gated(a, w, outs[1])
                        got.append(outs)
                finally:
                    kernels.gemm_bf16_force_tiling(-1)
                assert all(torch.equal(x, y) for x, y in zip(*got)), (m, n, k, ranges)
                assert _rel(got[0][0], a.double() @ w.double().T) < 1e-5


@pytest.mark.parametrize("rows,tiling", [(32, 21), (96, 21), (64 * 256, 21), (64 * 256 + 32, 22), (96 * 256, 22), (96 * 256 + 32, 23),
                                         (128 * 256 + 32, 24), (160 * 256 + 32, 25), (224 * 256, 25), (224 * 256 + 32, 23)])
def test_gated_products_of_up_to_64_tokens_take_tiles_of_64_with_the_same_bits(rows, tiling):
    """At each width of a tile, its last number of weight rows and the next one's first: the bits of the 128x128 tiles, with and
    without the norm before the product, whichever of the LDS-shared kernel's plans asks."""
    from vipera_rs_amd.ops import kernels
    if kernels.compute_units(torch.device(DEV)) != 256:
        pytest.skip("the widths follow the number of CUs")
    for m, k in ((17, 64), (33, 192), (64, 320), (5, 128)):
        g = torch.Generator().manual_seed(rows + m)
        a = torch.randn(m, k, generator=g).to(torch.bfloat16).to(DEV)
        w = torch.randn(rows, k, generator=g).to(torch.bfloat16).to(DEV)
        groups, stride = 5, kernels.follow_stride(m)
        sumsq = (torch.rand(groups * stride, generator=g) * k / groups).to(DEV)
        assert kernels.gemm_bf16_tile_carried_out(m, rows, k, gated=True) == tiling
        got = []
        try:
            for forced in (-1, 9):
                kernels.gemm_bf16_force_tiling(forced)
                outs = [torch.full((m, rows // 2), 7.0, dtype=torch.bfloat16, device=DEV) for _ in range(4)]
                kernels.gemm_bf16_gated(a, w, outs[0], 3)
                kernels.gemm_bf16_gated_tile_scaled(a, w, outs[1], sumsq, groups, 1e-5)
                for plan in (1, 2):
                    kernels.gemm_bf16_gated(a, w, outs[1 + plan], plan)
                got.append(outs)
        finally:
            kernels.gemm_bf16_force_tiling(-1)
        assert all(torch.equal(x, y) for x, y in zip(*got)) and torch.equal(got[0][0], got[0][2]) and torch.equal(got[0][0], got[0][3])
        product = a.double() @ w.double().T
        blocks = product.view(m, rows // 32, 2, 16)
        gate, up = blocks[:, :, 0].reshape(m, -1), blocks[:, :, 1].reshape(m, -1)
        assert _rel(got[0][0], up * gate / (1 + torch.exp(-gate))) < 8e-3


@pytest.mark.parametrize("rows,tiling", [(96, 21), (96 * 256, 22), (96 * 256 + 32, 23), (160 * 256, 24), (224 * 256, 25)])
@pytest.mark.parametrize("m,k", [(17, 320), (33, 1088), (64, 2112), (40, 768)])
def test_tiles_of_64_tokens_give_the_bits_of_the_kernel_that_shares_the_activations(rows, tiling, m, k):
    """That kernel takes up to 16 tokens at these K: every 16 tokens through it, K in several of its chunks of 256 and the rest of
    one, and of five to 33 steps of the tiles."""
    from vipera_rs_amd.ops import kernels
    if kernels.compute_units(torch.device(DEV)) != 256:
        pytest.skip("the widths follow the number of CUs")
    g = torch.Generator(DEV).manual_seed(rows + m)
    a = torch.randn(m, k, generator=g, device=DEV).to(torch.bfloat16)
    w = torch.randn(rows, k, generator=g, device=DEV).to(torch.bfloat16)
    got = torch.full((m, rows // 2), 7.0, dtype=torch.bfloat16, device=DEV)
    kernels.gemm_bf16_gated(a, w, got, 1)
    assert kernels.gemm_bf16_tile_launched()[0] == tiling
    for plan in (1, 2):
        shared = torch.full((m, rows // 2), 7.0, dtype=torch.bfloat16, device=DEV)
        for first in range(0, m, 16):
            kernels.gemm_bf16_gated(a[first:first + 16], w, shared[first:first + 16], plan)
        assert torch.equal(got, shared), plan


@pytest.mark.parametrize("plan", [1, 2])
@pytest.mark.parametrize("m,rows,k", [(24, 512, 2048), (33, 1056, 2048), (49, 96, 4096), (64, 8192, 2048), (64, 544, 264), (20, 160, 1032),
                                      (48, 64, 520)])
def test_the_kernel_that_shares_the_activations_takes_17_to_64_tokens_where_tiles_do_not(m, rows, k, plan):
    """K a multiple of 2,048, where its workgroups start at chunks of their own, and K in no whole steps of 64: two to four blocks of
    16 tokens give the bits of one block at a time, and 64-bit."""
    from vipera_rs_amd.ops import kernels
    g = torch.Generator(DEV).manual_seed(rows + m)
    a = torch.randn(m, k, generator=g, device=DEV).to(torch.bfloat16)
    w = torch.randn(rows, k, generator=g, device=DEV).to(torch.bfloat16)
    out, blocks = (torch.full((m, rows // 2), 7.0, dtype=torch.bfloat16, device=DEV) for _ in range(2))
    before = kernels.gemm_bf16_tile_launched()
    kernels.gemm_bf16_gated(a, w, out, plan)
    for first in range(0, m, 16):
        kernels.gemm_bf16_gated(a[first:first + 16], w, blocks[first:first + 16], plan)
    assert kernels.gemm_bf16_tile_launched() == before          # no tile ran
    assert torch.equal(out, blocks)
    gate, up = (a.double() @ w.double().T).view(m, rows // 32, 2, 16).unbind(2)
    gate, up = gate.reshape(m, -1), up.reshape(m, -1)
    assert _rel(out, up * gate / (1 + torch.exp(-gate))) < 8e-3


@pytest.mark.parametrize("tiling,other", [(5, 7), (6, 7), (9, 8)])
def test_tiles_with_a_third_stage_of_the_weight_divide_by_a_norm_with_the_bits_of_the_others(tiling, other):
    """The norm's sums follow the loop there, in LDS that held the stages: runs of K shorter than the stages, as long and longer,
    against the tiles of as many threads a token, which add them before it."""
    from vipera_rs_amd.ops import kernels
    g = torch.Generator().manual_seed(tiling)
    for m, rows in ((257, 288), (300, 416)):
        for k in (64, 128, 192, 256, 320, 1152):
            a = torch.randn(m, k, generator=g).to(torch.bfloat16).to(DEV)
            w = torch.randn(rows, k, generator=g).to(torch.bfloat16).to(DEV)
            for groups in (1, 7, 70):
                stride = kernels.follow_stride(m)
                sumsq = (torch.rand(groups * stride, generator=g) * k / groups).to(DEV)
                outs = [torch.full((m, rows // 2), 7.0, dtype=torch.bfloat16, device=DEV) for _ in range(2)]
                try:
                    for one, out in zip((tiling, other), outs):
                        kernels.gemm_bf16_force_tiling(one)
                        kernels.gemm_bf16_gated_tile_scaled(a, w, out, sumsq, groups, 1e-5)
                        assert kernels.gemm_bf16_tile_launched()[0] == one
                finally:
                    kernels.gemm_bf16_force_tiling(-1)
                assert torch.equal(*outs), (m, rows, k, groups)
                factor = 1 / torch.sqrt(sumsq.view(groups, stride)[:, :m].double().sum(0) / k + 1e-5)
                gate, up = (a.double() @ w.double().T * factor[:, None]).view(m, rows // 32, 2, 16).unbind(2)
                gate, up = gate.reshape(m, -1), up.reshape(m, -1)
                assert _rel(outs[0], up * gate / (1 + torch.exp(-gate))) < 8e-3


@pytest.mark.parametrize("m,n,k,tiling", [(1396, 1536, 1536, 16), (783, 4096, 2048, 17), (1000, 4608, 3584, 18), (2210, 4096, 1024, 19),
                                          (910, 9216, 2048, 20)])
def test_a_plan_of_one_range_is_carried_out_with_the_same_bits(m, n, k, tiling):
    from vipera_rs_amd.ops import kernels
    g = torch.Generator().manual_seed(m + n + k)
    a = torch.randn(m, k, generator=g).to(torch.bfloat16).to(DEV)
    w = torch.randn(n, k, generator=g).to(torch.bfloat16).to(DEV)
    assert kernels.gemm_bf16_tile_carried_out(m, n, k) == tiling
    out, other = torch.empty(m, n, device=DEV), torch.empty(m, n, device=DEV)
    kernels.gemm_bf16(a, w, None, out)
    assert kernels.gemm_bf16_tile_launched()[0] == tiling
    try:
        kernels.gemm_bf16_force_tiling(kernels.gemm_bf16_tile_plan(m, n, k)[0])
        kernels.gemm_bf16(a, w, None, other)
        assert kernels.gemm_bf16_tile_launched()[0] == kernels.gemm_bf16_tile_plan(m, n, k)[0]
    finally:
        kernels.gemm_bf16_force_tiling(-1)
    assert torch.equal(out, other)


@pytest.mark.parametrize("m,n,k,tiling,before,cut", [(1396, 1536, 8960, 20, 6, 4), (1201, 896, 4864, 18, 7, 4), (400, 900, 4864, 17, 9, 8),
                                                     (311, 3584, 4736, 18, 9, 4), (400, 4608, 3584, 18, 7, 2), (130, 5120, 13824, 20, 6, 8),
                                                     (311, 1024, 4096, 16, 13, 8), (200, 1530, 8960, 17, 13, 8), (622, 1536, 8960, 17, 14, 4),
                                                     (130, 3580, 3584, 16, 14, 4)])
def test_a_plan_of_several_ranges_is_carried_out_with_the_same_bits(m, n, k, tiling, before, cut):
    """The tile that is picked and the one of the estimate by whole rounds, with the same cut of K; results of either kind."""
    from vipera_rs_amd.ops import kernels
    g = torch.Generator().manual_seed(m + n + k)
    a = torch.randn(m, k, generator=g).to(torch.bfloat16).to(DEV)
    w = torch.randn(n, k, generator=g).to(torch.bfloat16).to(DEV)
    old = torch.randn(m, n, generator=g).to(DEV)
    for dtype, accumulate in ((torch.float32, False), (torch.bfloat16, False), (torch.float32, True)):
        out, other = old.to(dtype), old.to(dtype)
        kernels.gemm_bf16(a, w, None, out, accumulate)
        assert kernels.gemm_bf16_tile_launched()[:2] == (tiling, cut)
        try:
            kernels.gemm_bf16_force_tiling(before, cut)
            kernels.gemm_bf16(a, w, None, other, accumulate)
        finally:
            kernels.gemm_bf16_force_tiling(-1)
        assert torch.equal(out, other)


@pytest.mark.parametrize("m,n,k", [(399, 4288, 512), (288, 8320, 1024), (1435, 5440, 256), (695, 5440, 2048), (1805, 8896, 512),
                                   (512, 1056, 2048), (512, 64, 2048), (330, 7488, 7168), (100, 4608, 3584), (700, 4096, 2040)])
def test_a_product_launches_the_tile_that_the_plan_names_and_works_it_out_once(m, n, k):
    """For results of 32 and 16 bits, results added to what is there and gated ones, at sizes where these take different tiles,
    with and without ranges of K, up to 128 tokens and over a K of no whole steps of 64."""
    from vipera_rs_amd.ops import kernels
    g = torch.Generator().manual_seed(m + n + k)
    a = torch.randn(m, k, generator=g).to(torch.bfloat16).to(DEV)
    w = torch.randn(n, k, generator=g).to(torch.bfloat16).to(DEV)
    calls = [(4, False, lambda: kernels.gemm_bf16(a, w, None, torch.empty(m, n, device=DEV))),
             (2, False, lambda: kernels.gemm_bf16(a, w, None, torch.empty(m, n, dtype=torch.bfloat16, device=DEV))),
             (8, False, lambda: kernels.gemm_bf16(a, w, None, torch.zeros(m, n, device=DEV), accumulate=True)),
             (2, True, lambda: kernels.gemm_bf16_gated(a, w, torch.empty(m, n // 2, dtype=torch.bfloat16, device=DEV)))]
    for output_bytes, gated, call in calls:
        call()
        tiling, ranges, plans = kernels.gemm_bf16_tile_launched()
        assert tiling == kernels.gemm_bf16_tile_carried_out(m, n, k, gated, output_bytes), (output_bytes, gated)
        assert ranges == kernels.gemm_bf16_tile_plan(m, n, k, gated)[1], (output_bytes, gated)
        call()
        assert kernels.gemm_bf16_tile_launched() == (tiling, ranges, plans), "a plan kept for these sizes was worked out again"


@pytest.mark.parametrize("m,n,k,tiling", [(129, 33, 2048, 13), (512, 64, 2048, 13), (161, 1792, 10496, 13), (512, 2048, 512, 14),
                                          (512, 1057, 2048, 14), (468, 1792, 4352, 14), (512, 2576, 512, 15), (700, 5120, 2048, 15),
                                          (140, 5536, 1600, 15), (330, 7488, 7168, 9), (953, 512, 6400, 9)])
def test_the_tiles_chosen_for_a_product_do_not_change_its_bits(m, n, k, tiling):
    """Past 128 tokens a product planned as 128x128 tiles may be carried out by smaller ones: it is at these sizes, one beside
    each line of the choice, with the bits that the 128x128 tiles give with the planned ranges of K."""
    from vipera_rs_amd.ops import kernels
    g = torch.Generator().manual_seed(m + n + k)
    a = torch.randn(m, k, generator=g).to(torch.bfloat16).to(DEV)
    w = torch.randn(n, k, generator=g).to(torch.bfloat16).to(DEV)
    out, other = torch.empty(m, n, device=DEV), torch.empty(m, n, device=DEV)
    chosen, ranges = kernels.gemm_bf16_tile_plan(m, n, k)
    assert chosen == tiling
    kernels.gemm_bf16(a, w, None, out)
    assert _rel(out, a.double() @ w.double().T) < 1e-5
    try:
        kernels.gemm_bf16_force_tiling(9, ranges)
        kernels.gemm_bf16(a, w, None, other)
    finally:
        kernels.gemm_bf16_force_tiling(-1)
    assert torch.equal(out, other)
    if ranges > 1:      # and no other number of ranges gives them
        try:
            kernels.gemm_bf16_force_tiling(9, ranges // 2)
            kernels.gemm_bf16(a, w, None, other)
        finally:
            kernels.gemm_bf16_force_tiling(-1)
        assert not torch.equal(out, other)


@pytest.mark.parametrize("tiling", [0, 9, 7, 5, 6])
def test_the_tiled_kernel_computes_the_same_in_every_order_of_its_tiles(tiling):
    """The workgroups walk the tiles in blocks of a few rows of tiles (chosen by shape, forced here): every tile is
    computed once whatever the block height, also where the last block has fewer rows and where the launch has
    more workgroups than tiles."""
    from vipera_rs_amd.ops import kernels
    g = torch.Generator().manual_seed(tiling)
    m, n, k = 1100, 1300, 192
    a = torch.randn(m, k, generator=g).to(torch.bfloat16).to(DEV)
    w = torch.randn(n, k, generator=g).to(torch.bfloat16).to(DEV)
    want = a.double() @ w.double().T
    outs = []
    try:
        for ranges in (1, 3):
            kernels.gemm_bf16_force_tiling(tiling, ranges)
            for rows in (0, 1, 2, 4, 5, 7, 50):
                kernels.gemm_bf16_force_tile_group(rows)
                out = torch.full((m, n), 7.0, device=DEV)
                kernels.gemm_bf16(a, w, None, out)
                assert _rel(out, want) < 1e-5, (ranges, rows)
                outs.append(out)
            assert all(torch.equal(outs[0], o) for o in outs[1:]), ranges
            outs.clear()
    finally:
        kernels.gemm_bf16_force_tile_group(0)
        kernels.gemm_bf16_force_tiling(-1)


@pytest.mark.parametrize("tiling", [9, 8])
@pytest.mark.parametrize("ranges", [1, 3])
def test_gemm_bf16_direct_tilings_with_three_lds_stages(tiling, ranges):
    """The 128-token tilings of the kernel that loads straight into LDS, forced to three stages (what up to 128
    tokens take by themselves) at any number of tokens: one, two, three, four and many K steps, so that the run
    ends in each stage, with and without a step whose loads stay in flight."""
    from vipera_rs_amd.ops import kernels
    shapes = [(64, 520, 64), (100, 264, 128), (128, 300, 192), (257, 520, 256), (65, 2100, 4608), (33, 1028, 1600),
              (300, 131, 1024)]
    try:
        kernels.gemm_bf16_force_tiling(tiling, ranges, stages=3)
        for m, n, k in shapes:
            g = torch.Generator().manual_seed(m + n + k)
            a = torch.randn(m, k, generator=g).to(torch.bfloat16).to(DEV)
            w = torch.randn(n, k, generator=g).to(torch.bfloat16).to(DEV)
            bias = torch.randn(n, generator=g).to(DEV)
            product = a.double() @ w.double().T
            for out_dtype, tol in ((torch.float32, 1e-5), (torch.bfloat16, 6e-3)):
                out = torch.full((m, n), 7.0, dtype=out_dtype, device=DEV)
                kernels.gemm_bf16(a, w, bias, out, skinny_limit=0)
                assert _rel(out, product + bias.double()) < tol, (m, n, k, out_dtype)
            base = torch.randn(m, n, generator=g).to(DEV)
            acc = base.clone()
            kernels.gemm_bf16(a, w, None, acc, accumulate=True, skinny_limit=0)
            assert _rel(acc, base.double() + product) < 1e-5, (m, n, k, "accumulate")
    finally:
        kernels.gemm_bf16_force_tiling(-1)


@pytest.mark.parametrize("tiling,stages", [(t, 0) for t in (0, 2, 3, 4, 9, 7, 8, 5, 10, 11, 12)]   # the last three: 128 tokens x 96, 160, 224 rows
                         + [(t, 3) for t in (9, 8, 10, 11, 12)] + [(t, 2) for t in (9, 11)])
def test_gated_product_with_every_tiling(tiling, stages):
    from vipera_rs_amd.ops import kernels
    from vipera_rs_amd.ops.linear import interleave_gate_up
    try:
        kernels.gemm_bf16_force_tiling(tiling, 1, stages)
        for m, inter, k in [(300, 208, 192), (2048, 528, 128), (130, 1008, 640), (70, 48, 72), (64, 304, 3584), (17, 160, 64)]:
            g = torch.Generator().manual_seed(m + inter + k)
            a = torch.randn(m, k, generator=g).to(torch.bfloat16).to(DEV)
            gate = torch.randn(inter, k, generator=g).to(torch.bfloat16).to(DEV)
            up = torch.randn(inter, k, generator=g).to(torch.bfloat16).to(DEV)
            gd, ud = a.double() @ gate.double().T, a.double() @ up.double().T
            out = torch.full((m, inter), 7.0, dtype=torch.bfloat16, device=DEV)
            kernels.gemm_bf16_gated(a, interleave_gate_up(gate, up), out)
            assert _rel(out, ud * (gd / (1 + torch.exp(-gd)))) < 8e-3, (m, inter, k)
    finally:
        kernels.gemm_bf16_force_tiling(-1)


@pytest.mark.parametrize("m,n,k", [(1, 100, 64), (8, 4608, 256), (16, 333, 520), (3, 9, 128), (5, 47, 72)])
def test_skinny_product_with_every_number_of_rows_per_workgroup(m, n, k):
    """A workgroup of the weight-streaming kernel may own 8 to 16 weight rows; the launcher picks the number
    that divides N evenly over the CUs.  Every choice gives the same sums (the order within a row's sum does
    not depend on it), beside bias, accumulation and both output types."""
    from vipera_rs_amd.ops import kernels
    g = torch.Generator().manual_seed(m + n + k)
    a = torch.randn(m, k, generator=g).to(torch.bfloat16).to(DEV)
    w = torch.randn(n, k, generator=g).to(torch.bfloat16).to(DEV)
    bias = torch.randn(n, generator=g).to(DEV)
    base = torch.randn(m, n, generator=g).to(DEV)
    want = a.double() @ w.double().T + bias.double()
    first = {}
    for shape in [0] + list(range(108, 117)):
        out = torch.full((m, n), 7.0, dtype=torch.bfloat16, device=DEV)
        kernels.gemm_bf16(a, w, bias, out, skinny_shape=shape)
        assert _rel(out, want) < 6e-3, shape
        acc = base.clone()
        kernels.gemm_bf16(a, w, bias, acc, accumulate=True, skinny_shape=shape)
        assert _rel(acc, base.double() + want) < 1e-5, shape
        if first:
            assert torch.equal(out, first["out"]) and torch.equal(acc, first["acc"]), shape
        first = first or {"out": out, "acc": acc}



def test_gemm_bf16_tile_and_skinny_kernels_agree():
    from vipera_rs_amd.ops import kernels
    g = torch.Generator().manual_seed(5)
    a = torch.randn(48, 256, generator=g).to(torch.bfloat16).to(DEV)
    w = torch.randn(272, 256, generator=g).to(torch.bfloat16).to(DEV)
    skinny = torch.empty(48, 272, dtype=torch.float32, device=DEV)
    tile = torch.empty_like(skinny)
    kernels.gemm_bf16(a, w, None, skinny, skinny_limit=64)
    kernels.gemm_bf16(a, w, None, tile, skinny_limit=0)
    assert _rel(skinny, tile) < 1e-5


def test_gemm_bf16_strided_views():
    from vipera_rs_amd.ops import kernels
    g = torch.Generator().manual_seed(9)
    wide = torch.randn(20, 96 + 64, generator=g).to(torch.bfloat16).to(DEV)
    a = wide[:, :96]
    w = torch.randn(40, 96, generator=g).to(torch.bfloat16).to(DEV)
    out_wide = torch.zeros(20, 100, dtype=torch.bfloat16, device=DEV)
    out = out_wide[:, 20:60]
    kernels.gemm_bf16(a, w, None, out)
    assert _rel(out, a.double() @ w.double().T) < 6e-3
    assert float(out_wide[:, :20].abs().max()) == 0.0 and float(out_wide[:, 60:].abs().max()) == 0.0


@pytest.mark.parametrize("m,n,k", [(1, 48, 64), (7, 300, 96), (65, 130, 71), (130, 67, 200)])
@pytest.mark.parametrize("dtypes", [(torch.float32,) * 3, (torch.bfloat16, torch.float32, torch.bfloat16),
                                    (torch.bfloat16, torch.bfloat16, torch.float32)])
def test_gemm_generic_against_float64(m, n, k, dtypes):
    from vipera_rs_amd.ops import kernels
    g = torch.Generator().manual_seed(m + n + k)
    a = torch.randn(m, k, generator=g).to(dtypes[0]).to(DEV)
    w = torch.randn(n, k, generator=g).to(dtypes[1]).to(DEV)
    bias = torch.randn(n, generator=g).to(DEV)
    out = torch.empty(m, n, dtype=dtypes[2], device=DEV)
    kernels.gemm_generic(a, w, bias, out)
    want = a.double() @ w.double().T + bias.double()
    assert _rel(out, want) < (2e-6 if dtypes[2] == torch.float32 else 6e-3)


@pytest.mark.parametrize("k", [64, 200, 256, 1100, 2600])
def test_gemm_generic_does_not_depend_on_the_batch(k):
    """Every output element is summed in one fixed order (chains over ranges of 256 k, four ranges to a slab, slabs in
    ascending order), whichever kernel computes it: the weight stream that takes up to 8 tokens and the tiles that take 33 and
    64 give bit for bit the rows of the tiles that take 70, alone or in any company, with and without a bias, accumulating
    or not."""
    from vipera_rs_amd.ops import kernels
    g = torch.Generator().manual_seed(k)
    a = torch.randn(70, k, generator=g).to(DEV)
    w = torch.randn(90, k, generator=g).to(DEV)
    bias = torch.randn(90, generator=g).to(DEV)
    base = torch.randn(70, 90, generator=g).to(DEV)
    whole = torch.empty(70, 90, device=DEV)
    kernels.gemm_generic(a, w, None, whole)
    assert _rel(whole, a.double() @ w.double().T) < 2e-6
    for rows in ([37], [0, 1], list(range(5, 12)), list(range(50, 58)), list(range(61, 70)), list(range(3, 36)), list(range(6, 70))):
        part = torch.empty(len(rows), 90, device=DEV)
        kernels.gemm_generic(a[rows].contiguous(), w, None, part)
        assert torch.equal(part, whole[rows]), f"{len(rows)} rows"      # bit for bit
    with_bias = torch.empty(70, 90, device=DEV)
    kernels.gemm_generic(a, w, bias, with_bias)
    added = base.clone()
    kernels.gemm_generic(a, w, bias, added, accumulate=True)
    few = base[20:28].clone()
    kernels.gemm_generic(a[20:28], w, bias, few, accumulate=True)        # a view with a row stride of its own
    assert torch.equal(few, added[20:28])
    rounded = torch.empty(8, 90, dtype=torch.bfloat16, device=DEV)
    kernels.gemm_generic(a[20:28], w, bias, rounded)
    assert torch.equal(rounded, with_bias[20:28].to(torch.bfloat16))


@pytest.mark.parametrize("m,n,k", [(1024, 1024, 520), (1030, 1100, 1027), (1500, 905, 258), (1153, 1025, 2052)])
def test_many_tiles_of_gemm_generic_sum_in_the_same_order(m, n, k):
    """Against 64-bit, and bit for bit the rows that the tiles give 70 and 33 rows at a time and, where K is in fours, the weight
    stream 8 at a time; with a bias, accumulating, into bfloat16, from bfloat16 activations, and with rows that start off a
    16-byte boundary."""
    from vipera_rs_amd.ops import kernels
    g = torch.Generator().manual_seed(m + n + k)
    a = torch.randn(m, k, generator=g).to(DEV)
    w = torch.randn(n, k, generator=g).to(DEV)
    bias = torch.randn(n, generator=g).to(DEV)
    base = torch.randn(m, n, generator=g).to(DEV)
    whole = torch.full((m, n), float("nan"), device=DEV)
    kernels.gemm_generic(a, w, bias, whole)
    assert _rel(whole, a.double() @ w.double().T + bias.double()) < 2e-6
    for rows in (70, 33, 8):
        for start in (0, 128 * 3 + 5, m - rows):
            part = torch.empty(rows, n, device=DEV)
            kernels.gemm_generic(a[start:start + rows], w, bias, part)
            assert torch.equal(part, whole[start:start + rows]), (rows, start)       # bit for bit
    added = base.clone()
    kernels.gemm_generic(a, w, bias, added, accumulate=True)
    few = base[200:270].clone()
    kernels.gemm_generic(a[200:270], w, bias, few, accumulate=True)
    assert torch.equal(few, added[200:270])
    rounded = torch.empty(m, n, dtype=torch.bfloat16, device=DEV)
    kernels.gemm_generic(a, w, bias, rounded)
    assert torch.equal(rounded, whole.to(torch.bfloat16))
    half = a.to(torch.bfloat16)                                   # bfloat16 activations on a 32-bit weight
    mixed = torch.empty(m, n, device=DEV)
    kernels.gemm_generic(half, w, bias, mixed)
    again = torch.empty(m, n, device=DEV)
    kernels.gemm_generic(half.float(), w, bias, again)
    assert torch.equal(mixed, again)
    shifted = torch.zeros(m, k + 3, device=DEV)                   # rows 4 (k + 3) bytes apart, from a 4-byte offset
    shifted[:, 1:k + 1] = a
    out = torch.zeros(m, n + 8, device=DEV)
    kernels.gemm_generic(shifted[:, 1:k + 1], w, bias, out[:, 4:n + 4])
    assert torch.equal(out[:, 4:n + 4], whole)
    assert float(out[:, :4].abs().max()) == 0.0 and float(out[:, n + 4:].abs().max()) == 0.0


@pytest.mark.parametrize("m,n,k", [(9, 64, 256), (64, 65, 260), (65, 63, 1028), (200, 33, 3001), (1500, 1500, 1100), (1499, 1503, 2052),
                                   (2200, 2242, 1030)])
def test_gemm_generic_cut_over_workgroups_sums_in_the_same_order(m, n, k):
    """The tiled product with K whole, in slabs and in ranges, at sizes that end inside a tile, a step, a range and a slab:
    bit for bit the rows that the weight stream gives eight at a time, with a bias and accumulating; from 16-bit operands
    bit for bit what the same values give in 32-bit."""
    from vipera_rs_amd.ops import kernels
    g = torch.Generator().manual_seed(m + n + k)
    a, w = torch.randn(m, k, generator=g).to(DEV), torch.randn(n, k, generator=g).to(DEV)
    bias, base = torch.randn(n, generator=g).to(DEV), torch.randn(m, n, generator=g).to(DEV)
    whole, added = torch.full((m, n), float("nan"), device=DEV), base.clone()
    kernels.gemm_generic(a, w, bias, whole)
    kernels.gemm_generic(a, w, bias, added, accumulate=True)
    assert _rel(whole, a.double() @ w.double().T + bias.double()) < 2e-6
    padded = torch.nn.functional.pad(a, (0, -k % 4)), torch.nn.functional.pad(w, (0, -k % 4))   # the stream takes K in fours
    for start in (0, (m - 8) // 2, m - 8):
        rows = slice(start, start + 8)
        few, more = torch.empty(8, n, device=DEV), base[rows].clone()
        kernels.gemm_generic(padded[0][rows], padded[1], bias, few)
        kernels.gemm_generic(padded[0][rows], padded[1], bias, more, accumulate=True)
        assert torch.equal(few, whole[rows]) and torch.equal(more, added[rows]), start
    ha, hw = a.to(torch.bfloat16), w.to(torch.bfloat16)
    mixed, again = torch.empty(m, n, dtype=torch.bfloat16, device=DEV), torch.empty(m, n, device=DEV)
    kernels.gemm_generic(ha, hw, bias, mixed)
    kernels.gemm_generic(ha.float(), hw.float(), bias, again)
    assert torch.equal(mixed, again.to(torch.bfloat16))


@pytest.mark.parametrize("m,n,k,form", [(17, 33, 260, 1), (9, 1150, 896, 1), (16, 130, 4864, 1), (128, 1155, 1020, 2), (25, 1530, 8964, 2),
                                        (333, 1100, 1024, 3), (257, 1150, 516, 3), (64, 1536, 8964, 4), (260, 9731, 900, 5),
                                        (1000, 3001, 1028, 5), (65, 17930, 1540, 6), (400, 17921, 1036, 7), (2050, 6001, 260, 7)])
def test_each_form_of_the_32_bit_product_sums_in_the_same_order(m, n, k, form):
    """At sizes that take each kernel and end inside its tiles, steps, ranges and slabs: bit for bit the rows that the weight
    stream gives eight at a time, with a bias and accumulating; into and from rows of another stride, also where outputs do
    not lie on 16 bytes."""
    import ctypes
    from vipera_rs_amd.ops import kernels
    from vipera_rs_amd.ops.build import load_module
    chosen = load_module("gemm_generic").vk_gemm_generic_form
    chosen.argtypes, chosen.restype = [ctypes.c_int] * 3 + [ctypes.c_longlong], ctypes.c_int
    assert chosen(m, n, k, kernels._gemm_generic_parts(m, n, k)) == form
    g = torch.Generator(DEV).manual_seed(m + n + k)
    randn = lambda *shape: torch.randn(*shape, generator=g, device=DEV)
    strided, w, bias, base = randn(m, k + 4), randn(n, k), randn(n), randn(m, n)
    a = strided[:, :k]
    whole, added, wide = torch.full((m, n), float("nan"), device=DEV), base.clone(), torch.zeros(m, n + 9, device=DEV)
    kernels.gemm_generic(a, w, bias, whole)
    kernels.gemm_generic(a, w, bias, added, accumulate=True)
    kernels.gemm_generic(a.contiguous(), w, bias, wide[:, 4:n + 4])
    assert torch.equal(wide[:, 4:n + 4], whole) and float(wide[:, :4].abs().max()) == 0.0 and float(wide[:, n + 4:].abs().max()) == 0.0
    for start in (0, (m - 8) // 2, m - 8):
        rows = slice(start, start + 8)
        few, more = torch.empty(8, n, device=DEV), base[rows].clone()
        kernels.gemm_generic(a[rows], w, bias, few)
        kernels.gemm_generic(a[rows], w, bias, more, accumulate=True)
        assert torch.equal(few, whole[rows]) and torch.equal(more, added[rows]), start


@pytest.mark.parametrize("m,n,k,form", [(500, 130, 132, 1), (9, 33, 4, 1), (65, 4099, 132, 1), (17, 4099, 20, 2), (129, 2050, 4, 3), (257, 2050, 644, 9),
                                        (501, 2050, 644, 8), (65, 9731, 36, 6), (333, 9731, 100, 7), (33, 9731, 64, 5), (2003, 9731, 16, 0),
                                        (1001, 2050, 96, 0)])
def test_a_32_bit_product_of_short_rows_takes_the_form_that_is_fast_there(m, n, k, form):
    """Rows of less than 704 numbers, down to one step, beside each line of the choice (0: the 64 x 64 tiles)."""
    test_each_form_of_the_32_bit_product_sums_in_the_same_order(m, n, k, form)


@pytest.mark.parametrize("m,n,k,form", [(333, 9725, 900, 8), (39, 3037, 2052, 8), (35, 779, 11012, 8), (515, 1150, 900, 9),
                                        (36, 4979, 2052, 9), (333, 895, 4868, 9), (162, 4283, 1020, 4), (553, 105, 11012, 4)])
def test_wide_slabs_of_the_32_bit_product_sum_in_the_same_order(m, n, k, form):
    """The tiles of 48 x 48, 48 x 64 and 64 x 64 outputs over one slab and several, ending inside a tile, a step, a range and a
    slab, as their neighbours above."""
    test_each_form_of_the_32_bit_product_sums_in_the_same_order(m, n, k, form)


@pytest.mark.parametrize("k", [4, 200, 260, 1100])
@pytest.mark.parametrize("values", ["spread", "small operands", "small products", "small sums", "overflow", "special"])
def test_the_matrix_instruction_is_two_fused_multiply_adds_for_all_values(values, k):
    """The tiles on the matrix cores (70 rows) against the weight stream's FMA chains (8 rows at a time), bit for bit, NaN for
    NaN: magnitudes over the whole range of exponents, denormal operands, products and sums, overflow, infinities, NaN and
    zeros of both signs.  With one product per element both are the product rounded once, denormal results included."""
    from vipera_rs_amd.ops import kernels
    g = torch.Generator().manual_seed(k)
    scale = lambda rows, low, high: 2.0 ** torch.randint(low, high, (rows, k), generator=g).double()
    a, w = torch.randn(70, k, generator=g).double(), torch.randn(90, k, generator=g).double()
    exponents = {"spread": (-60, 60, -60, 60), "small operands": (-148, -126, 100, 126), "small products": (-80, -60, -80, -60),
                 "small sums": (-68, -65, -68, -65), "overflow": (50, 66, 50, 66), "special": (-3, 3, -3, 3)}[values]
    a, w = (a * scale(70, *exponents[:2])).float(), (w * scale(90, *exponents[2:])).float()
    if values == "special":
        for x, row in ((a, 5), (w, 7)):
            x[row, 0], x[row + 1, 1], x[row + 2, 2] = float("inf"), float("-inf"), float("nan")
            x[row + 3], x[row + 4], x[row + 5, 3] = 0.0, -0.0, 3.4e38
    if k == 4:
        a[:, 1:], w[:, 1:] = 0.0, 0.0          # one product per element
    a, w = a.to(DEV), w.to(DEV)
    tiles, stream = torch.empty(70, 90, device=DEV), torch.empty(70, 90, device=DEV)
    kernels.gemm_generic(a, w, None, tiles)
    for first in range(0, 70, 7):
        kernels.gemm_generic(a[first:first + 7], w, None, stream[first:first + 7])
    nan = torch.isnan(stream)
    bits = lambda x: x.masked_fill(torch.isnan(x), 0.0).view(torch.int32)
    assert torch.equal(torch.isnan(tiles), nan) and torch.equal(bits(tiles), bits(stream))
    if values.startswith("small"):
        denormal = a if values == "small operands" else stream
        assert bool(((denormal != 0.0) & (denormal.abs() < 2.0 ** -126)).any())
    if k == 4 and values != "special":
        assert torch.equal(tiles, (a[:, :1].double() * w[:, :1].double().T).float())


def test_cut_products_in_a_captured_step():
    """Products whose K is cut, one behind the other in a graph: their parts come from the graph's memory, and every replay gives
    the eager bits whatever the program allocates and computes in between."""
    from vipera_rs_amd.ops import kernels
    g = torch.Generator().manual_seed(8)
    a, w0 = torch.randn(24, 1100, generator=g).to(DEV), torch.randn(900, 1100, generator=g).to(DEV)
    w1, x = torch.randn(1100, 900, generator=g).to(DEV) / 30, torch.empty_like(a)
    assert kernels._gemm_generic_parts(24, 900, 1100) and kernels._gemm_generic_parts(24, 1100, 900)

    def step():
        x.copy_(a)
        for _ in range(3):
            hidden = torch.empty(24, 900, device=DEV)
            kernels.gemm_generic(x, w0, None, hidden)
            kernels.gemm_generic(hidden, w1, None, x, accumulate=True)

    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        step()
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        step()
    for turn in range(4):
        a.normal_()
        step()
        torch.cuda.synchronize()
        want = x.clone()
        x.fill_(float("nan"))
        noise = [torch.full((24, 900, 5), float(turn), device=DEV) for _ in range(4)]
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(x, want), turn
        del noise


def test_gemm_generic_needs_no_memory_for_its_parts():
    """Where the memory for the parts of a cut K is not there, the product runs uncut: the same bits."""
    from vipera_rs_amd.ops import kernels
    g = torch.Generator().manual_seed(3)
    a, w = torch.randn(128, 16384, generator=g).to(DEV), torch.randn(1024, 16384, generator=g).to(DEV)
    want, out = torch.empty(128, 1024, device=DEV), torch.full((128, 1024), float("nan"), device=DEV)
    assert kernels._gemm_generic_parts(128, 1024, 16384) == 64 * 128 * 1024
    kernels.gemm_generic(a, w, None, want)
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    room = torch.cuda.memory_reserved(DEV) + 2 ** 22      # the parts are 32 MB
    try:
        torch.cuda.set_per_process_memory_fraction(room / torch.cuda.get_device_properties(0).total_memory, 0)
        kernels.gemm_generic(a, w, None, out)
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0, 0)
    assert torch.equal(out, want)


@pytest.mark.parametrize("m,n,k,slabs", [(333, 1152, 896, 0), (64, 1536, 8960, 9), (65, 17930, 1540, 0), (333, 1152, 1100, 2)])
def test_a_32_bit_product_allocates_no_more_than_it_writes(m, n, k, slabs):
    """With that memory, and with all that any types would take, the same form and the same bits; with less it is refused."""
    import ctypes
    from vipera_rs_amd.ops import kernels
    from vipera_rs_amd.ops.build import load_module
    g = torch.Generator(DEV).manual_seed(m + n + k)
    a, w = torch.randn(m, k, generator=g, device=DEV), torch.randn(n, k, generator=g, device=DEV)
    out, all_parts = torch.empty(m, n, device=DEV), torch.empty(kernels._gemm_generic_parts(m, n, k), device=DEV)
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    torch.cuda.reset_peak_memory_stats()
    before = torch.cuda.memory_allocated()
    kernels.gemm_generic(a, w, None, out)
    assert torch.cuda.max_memory_allocated() - before <= slabs * m * n * 4 + 512
    lib, other = load_module("gemm_generic"), torch.empty(m, n, device=DEV)
    chosen = lib.vk_gemm_generic_form
    chosen.argtypes, chosen.restype = [ctypes.c_int] * 3 + [ctypes.c_longlong], ctypes.c_int
    assert chosen(m, n, k, slabs * m * n) == chosen(m, n, k, all_parts.numel())
    p, split = ctypes.c_void_p, lib.vk_gemm_generic_split
    def with_floats(floats):
        return split(p(a.data_ptr()), 0, p(w.data_ptr()), 0, p(0), p(other.data_ptr()), 0, m, n, k, ctypes.c_longlong(k), ctypes.c_longlong(n), 0,
                     p(all_parts.data_ptr()), ctypes.c_longlong(floats), p(torch.cuda.current_stream().cuda_stream))
    assert with_floats(all_parts.numel()) == 0
    torch.cuda.synchronize()
    assert torch.equal(out, other)
    assert not slabs or with_floats(slabs * m * n - 1) != 0


def test_gemm_generic_of_more_tiles_than_one_launch_takes():
    """Past 2^32 threads in its tiles a product is several launches: 1,048,576 x 65,600 outputs, 138 GB in bfloat16."""
    from vipera_rs_amd.ops import kernels
    torch.cuda.empty_cache()
    if torch.cuda.mem_get_info(DEV)[0] < 150e9:
        pytest.skip("needs 138 GB of free device memory for its output")
    m, n = 1048576, 65600
    a = (torch.arange(m, device=DEV) % 251 - 125).float()[:, None]      # whole numbers, and products below 2^8 times a power of two
    w = 2.0 ** (torch.arange(n, device=DEV) % 13 - 6).float()[:, None]
    out = torch.empty(m, n, dtype=torch.bfloat16, device=DEV)
    try:
        kernels.gemm_generic(a, w, None, out)
        for rows in (slice(0, 3), slice(m // 2, m // 2 + 3), slice(m - 3, m)):
            assert torch.equal(out[rows], (a[rows] * w.T).to(torch.bfloat16))
        for columns in (slice(0, 70), slice(n // 2, n // 2 + 70), slice(n - 200, n)):
            assert torch.equal(out[:, columns], (a * w[columns].T).to(torch.bfloat16))
    finally:
        del out
        torch.cuda.empty_cache()


@pytest.mark.parametrize("m,n,k", [(1, 64, 4), (2, 200, 520), (3, 70, 36), (4, 1000, 4096), (5, 129, 1028), (7, 333, 2052), (8, 3584, 1536)])
def test_gemm_stream_against_float64(m, n, k):
    """The 32-bit weight stream at sizes of its own: K that ends inside a chunk of 32, a range and a slab, rows of
    W that do not fill a workgroup's 64, every count of tokens' class, filled and not."""
    from vipera_rs_amd.ops import kernels
    g = torch.Generator().manual_seed(m * n + k)
    a = torch.randn(m, k, generator=g).to(DEV)
    w = torch.randn(n, k, generator=g).to(DEV)
    bias = torch.randn(n, generator=g).to(DEV)
    out = torch.full((m, n), float("nan"), device=DEV)
    kernels.gemm_generic(a, w, bias, out)
    assert _rel(out, a.double() @ w.double().T + bias.double()) < 2e-6
    wide = torch.zeros(m, n + 8, device=DEV)                               # an output with a row stride of its own
    kernels.gemm_generic(a, w, None, wide[:, 4:n + 4])
    assert _rel(wide[:, 4:n + 4], a.double() @ w.double().T) < 2e-6
    assert float(wide[:, :4].abs().max()) == 0.0 and float(wide[:, n + 4:].abs().max()) == 0.0


# --- attention -------------------------------------------------------------------------------------
def _plain_attention(q, k, v, first_pos, window, scale):
    """q: [T, heads, hd] at positions first_pos..; k, v: [P, kv_heads, hd] for positions 0..P-1. float64."""
    T, heads, hd = q.shape
    group = heads // k.shape[1]
    out = torch.zeros(T, heads, hd, dtype=torch.float64)
    for t in range(T):
        pos = first_pos + t
        lo = max(0, pos + 1 - window) if window > 0 else 0
        for h in range(heads):
            kk, vv = k[lo:pos + 1, h // group], v[lo:pos + 1, h // group]
            w = torch.softmax((kk @ q[t, h]) * scale, dim=0)
            out[t, h] = w @ vv
    return out


class _Paged:
    """A paged cache filled by hand: shuffled pages, K [page, kvh, slot, hd], V [page, kvh, hd, slot]."""

    def __init__(self, seqs, kv_heads, hd, block_size, dtype, seed, stale_nan=False):
        g = torch.Generator().manual_seed(seed)
        self.block_size = block_size
        need = [(n + block_size - 1) // block_size for n in seqs]
        pages = sum(need) + 3
        order = torch.randperm(pages, generator=g).tolist()
        self.k = (torch.randn(pages, kv_heads, block_size, hd, generator=g) * 7).to(dtype)   # stale values everywhere
        self.v = (torch.randn(pages, kv_heads, hd, block_size, generator=g) * 7).to(dtype)
        if stale_nan:
            # what no live position occupies is not finite, as after a request whose activations overflowed gave its
            # pages back: also the slots of a held page past the request's last position
            self.k.fill_(float("nan"))
            self.v.fill_(float("nan"))
        self.tables, self.keys, self.values = [], [], []
        for n, blocks in zip(seqs, need):
            table = [order.pop() for _ in range(blocks)]
            keys = torch.randn(n, kv_heads, hd, generator=g).to(dtype)
            values = torch.randn(n, kv_heads, hd, generator=g).to(dtype)
            whole, rest = n // block_size, n % block_size       # position p sits in slot p % size of page table[p // size]
            if whole:
                pages_of = torch.tensor(table[:whole])
                self.k[pages_of] = keys[:whole * block_size].view(whole, block_size, kv_heads, hd).permute(0, 2, 1, 3)
                self.v[pages_of] = values[:whole * block_size].view(whole, block_size, kv_heads, hd).permute(0, 2, 3, 1)
            if rest:
                self.k[table[whole], :, :rest, :] = keys[whole * block_size:].permute(1, 0, 2)
                self.v[table[whole], :, :, :rest] = values[whole * block_size:].permute(1, 2, 0)
            self.tables.append(table)
            self.keys.append(keys)
            self.values.append(values)
        width = max(need)
        self.table = torch.full((len(seqs), width), -1, dtype=torch.int32)
        for i, t in enumerate(self.tables):
            self.table[i, :len(t)] = torch.tensor(t, dtype=torch.int32)
        self.spare = order.pop()        # a page that no request holds

    def with_pages_given_back(self, first_visible):
        """The table after a window has passed: the blocks of entry i that lie wholly before position
        ``first_visible[i]`` name a page that nobody holds (in the engine their id is -1, which must not be followed;
        a kernel that reads such a block here reads what the spare page holds, NaN in the tests that say so)."""
        table = self.table.clone()
        for i, first in enumerate(first_visible):
            table[i, :first // self.block_size] = self.spare
        return table


ATTN_CASES = [
    # heads, kv_heads, hd, block_size, window, entries as (kv length after the step, tokens in the step)
    (4, 2, 16, 16, 0, [(37, 37), (70, 1), (5, 2)]),
    (3, 1, 32, 8, 21, [(90, 17), (64, 1), (33, 33), (130, 1)]),
    (6, 3, 48, 16, 0, [(100, 64), (65, 65)]),
    (28, 4, 128, 16, 0, [(300, 1), (257, 130), (31, 1)]),
    (20, 1, 80, 32, 50, [(200, 1), (97, 96)]),
    (2, 2, 256, 64, 0, [(129, 1), (70, 70)]),
    # widths that fill their padded width with pages that divide 64: prompts go through the kernel that loads into LDS directly
    (8, 2, 64, 8, 40, [(200, 150), (64, 64), (300, 1), (391, 130)]),
    (4, 4, 128, 32, 100, [(333, 300), (128, 128), (2, 2)]),
    (5, 5, 64, 64, 0, [(190, 190), (321, 129)]),
    (2, 1, 256, 16, 70, [(260, 200)]),
]


@pytest.mark.parametrize("case", ATTN_CASES, ids=[f"h{c[0]}kv{c[1]}d{c[2]}b{c[3]}w{c[4]}" for c in ATTN_CASES])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("stale", ["finite", "nan"])
def test_attention_kernels_against_plain_softmax(case, dtype, stale):
    """``stale``: what the pool holds wherever no live position lies, the rest of a request's last page included:
    large finite numbers, or NaN (a weight of zero times NaN is NaN on the matrix cores, so such a slot must not
    reach a product at all)."""
    from vipera_rs_amd.ops import kernels
    from vipera_rs_amd.ops.attention import decode_chunking
    heads, kv_heads, hd, bs, window, entries = case
    scale = 1.0 / math.sqrt(hd)
    cache = _Paged([kv for kv, _ in entries], kv_heads, hd, bs, dtype, seed=heads * 100 + hd, stale_nan=stale == "nan")
    g = torch.Generator().manual_seed(hd)
    counts = [n for _, n in entries]
    T = sum(counts)
    width = (heads + 2 * kv_heads) * hd
    qkv = torch.randn(T, width, generator=g).to(dtype)
    starts = [0]
    for n in counts:
        starts.append(starts[-1] + n)
    first = [kv - n for kv, n in entries]
    positions = torch.tensor([first[e] + i for e, n in enumerate(counts) for i in range(n)], dtype=torch.int32)
    entry_of = torch.tensor([e for e, n in enumerate(counts) for _ in range(n)], dtype=torch.int32)
    want = torch.zeros(T, heads, hd, dtype=torch.float64)
    for e, (kv, n) in enumerate(entries):
        q = qkv[starts[e]:starts[e + 1], :heads * hd].double().view(n, heads, hd)
        want[starts[e]:starts[e + 1]] = _plain_attention(q, cache.keys[e].double(), cache.values[e].double(),
                                                         first[e], window, scale)
    want = want.view(T, heads * hd)
    dev = lambda t: t.to(DEV)  # noqa: E731
    # with a window, the pages that the first token of an entry no longer sees have been given back
    table = cache.with_pages_given_back([max(0, first[e] + 1 - window) for e in range(len(entries))]) if window else cache.table
    qkv_d, k_d, v_d, table_d = dev(qkv), dev(cache.k), dev(cache.v), dev(table)
    tol = 2e-6 if dtype == torch.float32 else 1.2e-2

    out = torch.zeros(T, heads * hd, dtype=dtype, device=DEV)
    kernels.attn_generic(qkv_d, k_d, v_d, out, dev(positions), dev(entry_of), table_d, heads, kv_heads, hd, scale, window)
    assert _rel(out.cpu(), want) < tol, "32-bit-arithmetic kernel"

    if dtype == torch.float32 and kernels.attn_decode_f32_supported(qkv_d, k_d, hd):
        # single tokens on the 32-bit kernel that splits their positions, the portions on the general one
        singles = [e for e, n in enumerate(counts) if n == 1]
        es = dev(torch.tensor(starts, dtype=torch.int32))
        fp = dev(torch.tensor(first, dtype=torch.int32))
        out3 = torch.zeros(T, heads * hd, dtype=dtype, device=DEV)
        if singles:
            chunks = (max(entries[e][0] for e in singles) + 255) // 256 + 1      # a chunk that sees nothing, too
            partial = torch.full((len(singles) * heads * chunks * (hd + 2),), float("nan"), device=DEV)
            kernels.attn_decode_f32(qkv_d, k_d, v_d, out3, partial, dev(torch.tensor(singles, dtype=torch.int32)), es, fp,
                                    table_d, heads, kv_heads, hd, scale, window, chunks)
        kernels.attn_generic(qkv_d, k_d, v_d, out3, dev(positions), dev(entry_of), table_d, heads, kv_heads, hd, scale, window,
                             skip_single_of=es)
        assert _rel(out3.cpu(), want) < tol, "32-bit decode kernel beside the general one"
        if kernels.attn_prefill_f32_supported(qkv_d, k_d, hd):
            # the portions on the 32-bit kernel that walks the positions in tiles; tiles of 128 or of 64 tokens
            for tile_tokens in (128, 64):
                tiles = [x for e, n in enumerate(counts) if n > 1 for off in range(0, n, tile_tokens) for x in (e, off)]
                rows = [t for e, n in enumerate(counts) if n > 1 for t in range(starts[e], starts[e + 1])]
                out4 = torch.full((T, heads * hd), float("nan"), dtype=dtype, device=DEV)
                kernels.attn_prefill_f32(qkv_d, k_d, v_d, out4, dev(torch.tensor(tiles, dtype=torch.int32)), tile_tokens, es,
                                         fp, table_d, heads, kv_heads, hd, scale, window)
                assert _rel(out4.cpu()[rows], want[rows]) < tol, f"32-bit prompt kernel, tiles of {tile_tokens}"
                others = [t for t in range(T) if t not in set(rows)]
                assert bool(torch.isnan(out4.cpu()[others]).all()), "the prompt kernel wrote a single token's row"

    if dtype == torch.bfloat16:
        from vipera_rs_amd.engine.batch import TILE_TOKENS
        tiles = [x for e, n in enumerate(counts) if n > 1 for off in range(0, n, TILE_TOKENS) for x in (e, off)]
        singles = [e for e, n in enumerate(counts) if n == 1]
        out2 = torch.zeros(T, heads * hd, dtype=dtype, device=DEV)
        es, fp = dev(torch.tensor(starts, dtype=torch.int32)), dev(torch.tensor(first, dtype=torch.int32))
        if tiles:
            halved = torch.zeros(T, heads * hd, dtype=dtype, device=DEV)   # a tile's positions halved between sixteen waves
            kernels.attn_bf16_prefill(qkv_d, k_d, v_d, halved, dev(torch.tensor(tiles, dtype=torch.int32)), es, fp,
                                      table_d, heads, kv_heads, hd, scale, window, split=True)
            rows = [t for e, n in enumerate(counts) if n > 1 for t in range(starts[e], starts[e + 1])]
            assert _rel(halved.cpu()[rows], want[rows]) < tol, "matrix-core prompt kernel, halved"
            reach = max(kv for kv, n in entries if n > 1)
            for chunk_tiles in (1, 2):          # a tile's positions in chunks of 64 and of 128, merged by a second kernel
                chunked = torch.zeros(T, heads * hd, dtype=dtype, device=DEV)
                kernels.attn_bf16_prefill(qkv_d, k_d, v_d, chunked, dev(torch.tensor(tiles, dtype=torch.int32)), es, fp,
                                          table_d, heads, kv_heads, hd, scale, window, chunk_tiles=chunk_tiles,
                                          max_chunks=-(-((reach + 63) // 64) // chunk_tiles))
                assert _rel(chunked.cpu()[rows], want[rows]) < tol, f"matrix-core prompt kernel, chunks of {chunk_tiles}"
            kernels.attn_bf16_prefill(qkv_d, k_d, v_d, out2, dev(torch.tensor(tiles, dtype=torch.int32)), es, fp,
                                      table_d, heads, kv_heads, hd, scale, window)
        if singles:
            longest = max(entries[e][0] for e in singles)
            for chunk, chunks in {decode_chunking(longest, len(singles), kv_heads, (heads // kv_heads + 15) // 16),
                                  (32, (longest + 31) // 32), (512, (longest + 511) // 512),
                                  (2048, (longest + 2047) // 2048)}:
                partial = torch.empty(len(singles) * heads * chunks * (hd + 2), device=DEV)
                kernels.attn_bf16_decode(qkv_d, k_d, v_d, out2, partial, dev(torch.tensor(singles, dtype=torch.int32)),
                                         es, fp, table_d, heads, kv_heads, hd, scale, window, chunk, chunks)
                assert _rel(out2.cpu(), want) < tol, f"matrix-core kernels, chunk {chunk}"
                if chunks <= kernels.ATTN_DECODE_JOINED_CHUNKS:   # a workgroup that takes all chunks and merges them itself
                    joined = out2.clone()
                    joined[[starts[e] for e in singles]] = 7.0
                    kernels.attn_bf16_decode(qkv_d, k_d, v_d, joined, None, dev(torch.tensor(singles, dtype=torch.int32)),
                                             es, fp, table_d, heads, kv_heads, hd, scale, window, chunk, chunks, join=True)
                    assert _rel(joined.cpu(), want) < tol, f"matrix-core kernels, chunk {chunk}, joined"
        assert _rel(out2.cpu(), want) < tol, "matrix-core kernels"


@pytest.mark.parametrize("window", [0, 1500])
def test_decode_attention_over_thousands_of_positions(window):
    """Single-token entries with long histories: many chunks, chunks that span more pages than a wave
    keeps ids of in a register (the table is then read step by step), chunks cut by a window's edge."""
    from vipera_rs_amd.ops import kernels
    heads, kv_heads, hd, bs = 8, 2, 64, 16
    lengths = [5000, 3333, 1, 4097]
    scale = 1.0 / math.sqrt(hd)
    dtype = torch.bfloat16
    cache = _Paged(lengths, kv_heads, hd, bs, dtype, seed=11)
    g = torch.Generator().manual_seed(5)
    qkv = torch.randn(len(lengths), (heads + 2 * kv_heads) * hd, generator=g).to(dtype)
    first = [n - 1 for n in lengths]
    want = torch.zeros(len(lengths), heads, hd, dtype=torch.float64)
    for e, n in enumerate(lengths):
        q = qkv[e:e + 1, :heads * hd].double().view(1, heads, hd)
        want[e] = _plain_attention(q, cache.keys[e].double(), cache.values[e].double(), first[e], window, scale)[0]
    want = want.view(len(lengths), heads * hd)
    dev = lambda t: t.to(DEV)  # noqa: E731
    qkv_d, k_d, v_d, table_d = dev(qkv), dev(cache.k), dev(cache.v), dev(cache.table)
    es = dev(torch.arange(len(lengths) + 1, dtype=torch.int32))
    fp = dev(torch.tensor(first, dtype=torch.int32))
    singles = dev(torch.arange(len(lengths), dtype=torch.int32))
    longest = max(lengths)
    for chunk in (128, 256, 1024, 4096):
        chunks = (longest + chunk - 1) // chunk
        out = torch.zeros(len(lengths), heads * hd, dtype=dtype, device=DEV)
        partial = torch.empty(len(lengths) * heads * chunks * (hd + 2), device=DEV)
        for dense in (False, True):
            out = torch.zeros(len(lengths), heads * hd, dtype=dtype, device=DEV)
            kernels.attn_bf16_decode(qkv_d, k_d, v_d, out, partial, singles, es, fp, table_d, heads, kv_heads, hd, scale,
                                     window, chunk, chunks, dense=dense)
            assert _rel(out.cpu(), want) < 1.2e-2, f"chunk {chunk}, dense {dense}"
            if chunks <= kernels.ATTN_DECODE_JOINED_CHUNKS:
                out = torch.zeros(len(lengths), heads * hd, dtype=dtype, device=DEV)
                kernels.attn_bf16_decode(qkv_d, k_d, v_d, out, None, singles, es, fp, table_d, heads, kv_heads, hd, scale,
                                         window, chunk, chunks, dense=dense, join=True)
                assert _rel(out.cpu(), want) < 1.2e-2, f"chunk {chunk}, dense {dense}, joined"


def _plain_attention_by_head(q, k, v, first_pos, window, scale):
    """The same as ``_plain_attention`` with one matrix of scores per head, for thousands of positions."""
    T, heads, hd = q.shape
    group = heads // k.shape[1]
    pos = first_pos + torch.arange(T)[:, None]
    key = torch.arange(k.shape[0])[None, :]
    visible = key <= pos
    if window > 0:
        visible &= key > pos - window
    out = torch.zeros(T, heads, hd, dtype=torch.float64)
    for h in range(heads):
        scores = (q[:, h] @ k[:, h // group].T) * scale
        out[:, h] = torch.softmax(scores.masked_fill(~visible, float("-inf")), dim=1) @ v[:, h // group]
    return out


def test_the_two_plain_attentions_agree():
    g = torch.Generator().manual_seed(0)
    q, k, v = (torch.randn(n, h, 16, generator=g, dtype=torch.float64) for n, h in ((5, 6), (40, 2), (40, 2)))
    for window in (0, 7):
        a = _plain_attention(q, k, v, 35, window, 0.25)
        b = _plain_attention_by_head(q, k, v, 35, window, 0.25)
        assert float((a - b).abs().max()) < 1e-12


BENCH_HEADS = [(28, 4, 128), (40, 8, 128), (12, 2, 128)]   # the 7B, 32B and 1.5B head shapes


def _context_bucket(kv_len):
    bucket = 256
    while bucket < kv_len:
        bucket *= 2
    return bucket


@pytest.mark.parametrize("heads,kv_heads,hd", BENCH_HEADS, ids=[f"h{h}kv{k}" for h, k, _ in BENCH_HEADS])
@pytest.mark.parametrize("batch", [8, 64])
def test_decode_attention_at_the_benchmark_head_shapes(heads, kv_heads, hd, batch):
    """Single-token entries at 4,096 and 3,000 positions (and a few short ones) in batches of 8 and 64, with the
    chunking the engine picks for the longest entry and for the context bucket a captured step is built for.
    In every entry one far key is made to stand out for the first head of each group, so that a chunk or a page
    that is dropped shows."""
    from vipera_rs_amd.ops import kernels
    from vipera_rs_amd.ops.attention import decode_chunking, joins_decode_chunks
    bs, scale, dtype = 16, 1.0 / math.sqrt(hd), torch.bfloat16
    lengths = [(4096, 3000, 2049, 4095, 1, 3001, 130, 4096)[e % 8] for e in range(batch)]
    if batch == 64 and heads != 28:
        # the other two head shapes at a quarter of the lengths: the float64 oracle is what the time goes to
        lengths = [(1024, 750, 513, 1023, 1, 751, 130, 1024)[e % 8] for e in range(batch)]
    cache = _Paged(lengths, kv_heads, hd, bs, dtype, seed=heads)
    g = torch.Generator().manual_seed(batch)
    qkv = torch.randn(batch, (heads + 2 * kv_heads) * hd, generator=g).to(dtype)
    group = heads // kv_heads
    for e, n in enumerate(lengths):
        far = (17 * (e + 1)) % n
        page, slot = cache.tables[e][far // bs], far % bs
        for kv in range(kv_heads):
            q = qkv[e, kv * group * hd:(kv * group + 1) * hd].float()
            key = (q / q.norm() * (9.0 / scale / q.norm())).to(dtype)      # a score of about 9 for that head
            cache.keys[e][far, kv] = key
            cache.k[page, kv, slot, :] = key
    first = [n - 1 for n in lengths]
    want = torch.zeros(batch, heads, hd, dtype=torch.float64)
    for e in range(batch):
        q = qkv[e:e + 1, :heads * hd].double().view(1, heads, hd)
        want[e] = _plain_attention_by_head(q, cache.keys[e].double(), cache.values[e].double(), first[e], 0, scale)[0]
    want = want.view(batch, heads * hd)
    dev = lambda t: t.to(DEV)  # noqa: E731
    qkv_d, k_d, v_d = dev(qkv), dev(cache.k), dev(cache.v)
    es = dev(torch.arange(batch + 1, dtype=torch.int32))
    fp = dev(torch.tensor(first, dtype=torch.int32))
    singles = dev(torch.arange(batch, dtype=torch.int32))
    longest = max(lengths)
    for visible in (longest, _context_bucket(longest), 2 * _context_bucket(longest)):
        # a captured step is built for a context bucket: its table is that wide and its chunks cover all of it
        width = (visible + bs - 1) // bs
        table = torch.full((batch, width), -1, dtype=torch.int32)
        table[:, :cache.table.shape[1]] = cache.table
        chunk, chunks = decode_chunking(visible, batch, kv_heads, (group + 15) // 16)
        out = torch.zeros(batch, heads * hd, dtype=dtype, device=DEV)
        partial = torch.full((batch * heads * chunks * (hd + 2),), float("nan"), device=DEV)
        kernels.attn_bf16_decode(qkv_d, k_d, v_d, out, partial, singles, es, fp, dev(table), heads, kv_heads, hd, scale, 0,
                                 chunk, chunks)
        assert _rel(out.cpu(), want) < 1.2e-2, f"visible {visible}: chunk {chunk} x {chunks}"
        # a step of single tokens only: the kernel is told that entry i is slot i and token i and looks neither up
        dense = torch.zeros(batch, heads * hd, dtype=dtype, device=DEV)
        kernels.attn_bf16_decode(qkv_d, k_d, v_d, dense, partial, singles, es, fp, dev(table), heads, kv_heads, hd, scale, 0,
                                 chunk, chunks, dense=True)
        assert torch.equal(dense, out)
        if joins_decode_chunks(chunks, batch, kv_heads, (group + 15) // 16, 256):   # what the engine does at batch 64
            joined = torch.zeros(batch, heads * hd, dtype=dtype, device=DEV)
            kernels.attn_bf16_decode(qkv_d, k_d, v_d, joined, None, singles, es, fp, dev(table), heads, kv_heads, hd, scale,
                                     0, chunk, chunks, dense=True, join=True)
            assert _rel(joined.cpu(), want) < 1.2e-2, f"visible {visible}: chunk {chunk} x {chunks}, joined"
    # the long chunks of many requests at long contexts, over a table as wide as theirs
    visible = 4 * _context_bucket(longest)
    table = torch.full((batch, (visible + bs - 1) // bs), -1, dtype=torch.int32)
    table[:, :cache.table.shape[1]] = cache.table
    for chunk in (2048, 4096):
        chunks = (visible + chunk - 1) // chunk
        out = torch.zeros(batch, heads * hd, dtype=dtype, device=DEV)
        partial = torch.full((batch * heads * chunks * (hd + 2),), float("nan"), device=DEV)
        kernels.attn_bf16_decode(qkv_d, k_d, v_d, out, partial, singles, es, fp, dev(table), heads, kv_heads, hd, scale, 0,
                                 chunk, chunks, dense=True)
        assert _rel(out.cpu(), want) < 1.2e-2, f"visible {visible}: chunk {chunk} x {chunks}"
        joined = torch.zeros(batch, heads * hd, dtype=dtype, device=DEV)
        kernels.attn_bf16_decode(qkv_d, k_d, v_d, joined, None, singles, es, fp, dev(table), heads, kv_heads, hd, scale,
                                 0, chunk, chunks, dense=True, join=True)
        assert _rel(joined.cpu(), want) < 1.2e-2, f"visible {visible}: chunk {chunk} x {chunks}, joined"
    out = torch.zeros(batch, heads * hd, dtype=dtype, device=DEV)
    kernels.attn_generic(qkv_d, k_d, v_d, out, fp, singles, dev(cache.table), heads, kv_heads, hd, scale, 0)
    assert _rel(out.cpu(), want) < 1.2e-2, "32-bit-arithmetic kernel on the bfloat16 cache"


@pytest.mark.parametrize("heads,kv_heads,hd,window,keep", [(14, 2, 64, 0, 0), (4, 1, 128, 0, 0), (8, 4, 128, 200, 70), (3, 3, 64, 96, 0)])
def test_prompt_tiles_shared_between_workgroups_and_narrow_addresses_give_the_same_bits(heads, kv_heads, hd, window, keep):
    """Tiles whose tokens end in the first and the second half, at a wave's edge and one past it, behind nothing and behind
    hundreds of positions; offsets of 32 bits against addresses of 64 for every form of the kernel."""
    from vipera_rs_amd.ops import kernels
    from vipera_rs_amd.ops.attention import AttentionExtras
    bs, dtype = 16, torch.bfloat16
    entries = [(2, 2), (64, 64), (65, 65), (500, 17), (900, 129), (333, 333), (1300, 208)]   # (positions after the step, tokens)
    cache = _Paged([kv for kv, _ in entries], kv_heads, hd, bs, dtype, seed=hd + heads)
    counts, first = [n for _, n in entries], [kv - n for kv, n in entries]
    starts = [sum(counts[:e]) for e in range(len(counts) + 1)]
    dev = lambda t: t.to(DEV)  # noqa: E731
    qkv = dev(torch.randn(starts[-1], (heads + 2 * kv_heads) * hd, generator=torch.Generator().manual_seed(heads)).to(dtype))
    tiles = sorted((first[e] + off, e, off) for e, n in enumerate(counts) for off in range(0, n, 128))
    arrays = [dev(torch.tensor(x, dtype=torch.int32)) for x in ([x for _, e, off in tiles for x in (e, off)], starts, first)]
    k, v, table = dev(cache.k), dev(cache.v), dev(cache.table)
    extras = AttentionExtras(keep_first=keep) if keep else None

    def run(split, pages, chunk_tiles=0, max_chunks=0):
        out = torch.full((starts[-1], heads * hd), 7.0, dtype=dtype, device=DEV)
        kernels.attn_bf16_prefill(qkv, k, v, out, *arrays, table, heads, kv_heads, hd, hd ** -0.5, window, split, chunk_tiles,
                                  max_chunks, extras=extras, cache_pages=pages)
        return out

    halved = run(1, None)
    assert torch.equal(run(2, None), halved) and torch.equal(run(2, 0), halved) and torch.equal(run(1, 0), halved)
    assert torch.equal(run(0, None), run(0, 0)) and torch.equal(run(0, None, 3, 8), run(0, 0, 3, 8))
    assert _rel(run(0, None), halved.double()) < 1.2e-2


# heads, kv_heads, hd, window, first positions kept, (positions after the step, tokens) of the prompts, positions of single tokens,
# whether sums may be reordered (no router), the prompts' (chunk, chunks; split), the single tokens' (chunk, chunks, joined)
DISPATCHED = [
    (16, 4, 128, 2048, 0, [(6000, 512)], [], True, ((6, 6), 0), None),          # cut by what the window leaves
    (16, 4, 128, 2048, 130, [(6000, 512)], [], True, ((7, 6), 0), None),
    (16, 4, 128, 2048, 0, [(6000, 512)], [], False, ((12, 8), 0), None),
    (4, 1, 256, -1500, 0, [(4000, 200)], [700], False, ((8, 8), 0), (128, 6, False)),
    (14, 2, 64, 0, 0, [(2000, 100)], [], True, ((4, 8), 0), None),
    (12, 2, 128, 0, 0, [(3000, 200), (700, 65)], [600, 40], True, ((4, 12), 0), (32, 19, False)),
    (8, 4, 128, 0, 0, [(333, 333), (200, 17)], [], True, (None, 2), None),      # halved and shared between two workgroups
    (3, 3, 64, 96, 70, [(500, 300), (65, 65)], [], False, (None, 2), None),
    (14, 2, 64, 0, 0, [], [512], True, None, (64, 8, True)),                    # short chunks, joined by the workgroup
    (14, 2, 64, 0, 0, [], [449, 1, 64, 65, 300], True, None, (64, 8, True)),
    (12, 2, 128, 150, 40, [], [256, 31, 129], True, None, (32, 8, True)),
    (28, 4, 128, 0, 0, [], [1000, 1, 33, 970, 64, 500, 999, 128], True, None, (64, 16, False)),
    (14, 2, 64, 200, 0, [], [1500, 3], True, None, (64, 24, False)),
]


@pytest.mark.parametrize("extended", [False, True], ids=["plain", "extended"])
@pytest.mark.parametrize("case", DISPATCHED, ids=[f"h{c[0]}d{c[2]}w{c[3]}-{i}" for i, c in enumerate(DISPATCHED)])
def test_paged_attention_with_the_plans_of_known_lengths_and_short_contexts(case, extended):
    """The dispatch over cut, halved and shared prompt tiles and over short decode chunks, of models with and without a router,
    against the kernel of 32-bit arithmetic; ``extended``: with a cap, a sink, a bias by distance and a gate."""
    from types import SimpleNamespace
    from vipera_rs_amd.ops import kernels
    from vipera_rs_amd.ops.attention import AttentionExtras, paged_attention
    heads, kv_heads, hd, window, keep, prompts, singles, free, prompt_plan, decode_plan = case
    entries = prompts + [(kv, 1) for kv in singles]
    cache = _Paged([kv for kv, _ in entries], kv_heads, hd, 16, torch.bfloat16, seed=hd + heads, stale_nan=True)
    counts, first = [n for _, n in entries], [kv - n for kv, n in entries]
    starts = [sum(counts[:e]) for e in range(len(counts) + 1)]
    g = torch.Generator().manual_seed(heads)
    qkv = torch.randn(starts[-1], (heads + 2 * kv_heads) * hd, generator=g).to(torch.bfloat16).to(DEV)
    ints = lambda v: torch.tensor(v, dtype=torch.int32, device=DEV)  # noqa: E731
    tiles = sorted((first[e] + off, e, off) for e, n in enumerate(counts) if n > 1 for off in range(0, n, 128))
    reaches = [pos + min(128, counts[e] - off) for pos, e, off in tiles]
    batch = SimpleNamespace(
        num_prefill_tiles=len(tiles), prefill_tiles=ints([x for _, e, off in tiles for x in (e, off)]), tile_reaches=reaches,
        max_tile_reach=max(reaches, default=0), sum_tile_reach=sum(reaches), entry_start=ints(starts), entry_first_pos=ints(first),
        num_decode_entries=len(singles), decode_entries=ints(list(range(len(prompts), len(entries)))), max_decode_kv_len=max(singles, default=0),
        sum_decode_kv_len=sum(singles), all_single=not prompts, shared={}, launch_plans=[], free_sum_order=free)
    table = cache.table
    if window and not keep:    # what the window has passed has been given back (a layer that keeps first positions keeps all pages)
        table = cache.with_pages_given_back([max(0, f + 1 - window) if window > 0 else f - f % -window for f in first])
    k, v, table = cache.k.to(DEV), cache.v.to(DEV), table.to(DEV)
    extras, cap = AttentionExtras(keep_first=keep), 0.0
    if extended:
        extras, cap = AttentionExtras(sink=torch.randn(heads, generator=g).to(DEV), rel=torch.randn(heads, 90, generator=g).to(DEV), keep_first=keep,
                                      gate=torch.randn(starts[-1], heads, generator=g).to(DEV)), 5.0
    want, got = (torch.full((starts[-1], heads * hd), 7.0, dtype=torch.bfloat16, device=DEV) for _ in range(2))
    kernels.attn_generic(qkv, k, v, want, ints([f + i for f, n in zip(first, counts) for i in range(n)]),
                         ints([e for e, n in enumerate(counts) for _ in range(n)]), table, heads, kv_heads, hd, hd ** -0.5, window,
                         softcap=cap, extras=extras)
    paged_attention(qkv, k, v, got, batch, table, heads, kv_heads, hd, hd ** -0.5, window, cap, extras)
    assert list(batch.shared.values()) == ([prompt_plan] if prompts else [])
    assert batch.launch_plans == ([decode_plan] if singles else [])
    for e in range(len(entries)):
        rows = slice(starts[e], starts[e + 1])
        assert _rel(got[rows], want[rows].double()) < 1.2e-2, entries[e]


@pytest.mark.parametrize("heads,kv_heads,hd", BENCH_HEADS, ids=[f"h{h}kv{k}" for h, k, _ in BENCH_HEADS])
def test_prompt_attention_at_the_benchmark_head_shapes(heads, kv_heads, hd):
    """One prompt of 2,048 tokens from position 0 and one portion of 512 tokens from position 3,584 in one step."""
    from vipera_rs_amd.engine.batch import TILE_TOKENS
    from vipera_rs_amd.ops import kernels
    bs, scale, dtype = 16, 1.0 / math.sqrt(hd), torch.bfloat16
    entries = [(2048, 2048), (4096, 512)]       # (positions in the cache after the step, tokens of the step)
    cache = _Paged([kv for kv, _ in entries], kv_heads, hd, bs, dtype, seed=hd + heads)
    g = torch.Generator().manual_seed(heads)
    counts = [n for _, n in entries]
    T = sum(counts)
    qkv = torch.randn(T, (heads + 2 * kv_heads) * hd, generator=g).to(dtype)
    starts, first = [0, counts[0], T], [kv - n for kv, n in entries]
    want = torch.zeros(T, heads, hd, dtype=torch.float64)
    for e, (kv, n) in enumerate(entries):
        q = qkv[starts[e]:starts[e + 1], :heads * hd].double().view(n, heads, hd)
        want[starts[e]:starts[e + 1]] = _plain_attention_by_head(q, cache.keys[e].double(), cache.values[e].double(),
                                                                 first[e], 0, scale)
    want = want.view(T, heads * hd)
    dev = lambda t: t.to(DEV)  # noqa: E731
    tiles = [(first[e] + off, e, off) for e, n in enumerate(counts) for off in range(0, n, TILE_TOKENS)]
    tiles = [x for _, e, off in sorted(tiles) for x in (e, off)]                # as the engine orders them
    # whole tiles, tiles in halves, and tiles in chunks of 8 and of 5 steps of 64 positions (the last chunk short)
    for split, chunk_tiles in ((False, 0), (True, 0), (False, 8), (False, 5)):
        out = torch.zeros(T, heads * hd, dtype=dtype, device=DEV)
        max_chunks = -(-(4096 // 64) // chunk_tiles) if chunk_tiles else 0
        kernels.attn_bf16_prefill(dev(qkv), dev(cache.k), dev(cache.v), out, dev(torch.tensor(tiles, dtype=torch.int32)),
                                  dev(torch.tensor(starts, dtype=torch.int32)), dev(torch.tensor(first, dtype=torch.int32)),
                                  dev(cache.table), heads, kv_heads, hd, scale, 0, split=split,
                                  chunk_tiles=chunk_tiles, max_chunks=max_chunks)
        got = out.cpu()
        assert _rel(got, want) < 1.2e-2, (split, chunk_tiles)
        # row by row too: the first tokens of a prompt see few keys, their outputs are large and would hide a fault
        # in a late row of small outputs
        rows = (got.double() - want).abs().amax(dim=1) / want.abs().amax(dim=1)
        assert float(rows.max()) < 3e-2, (split, chunk_tiles, int(rows.argmax()))


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_attention_finds_one_far_key_among_hundreds(dtype):
    """One early key is made to dominate: every later token must return (almost exactly) its value.
    An off-by-one in the visible range, a missed page or a wrong tile would lose it."""
    from vipera_rs_amd.ops import kernels
    heads, kv_heads, hd, bs, n = 4, 2, 64, 16, 700
    far = 17
    cache = _Paged([n], kv_heads, hd, bs, dtype, seed=1)
    direction = torch.randn(hd, generator=torch.Generator().manual_seed(3))
    direction = (direction / direction.norm()).to(dtype)
    page, slot = cache.tables[0][far // bs], far % bs
    cache.k[page, :, slot, :] = direction * 40
    q = torch.zeros(2, (heads + 2 * kv_heads) * hd, dtype=dtype)
    q[:, :heads * hd] = (direction * 40).repeat(heads)
    dev = lambda t: t.to(DEV)  # noqa: E731
    out = torch.zeros(2, heads * hd, dtype=dtype, device=DEV)
    positions = torch.tensor([n - 2, n - 1], dtype=torch.int32)
    kernels.attn_generic(dev(q), dev(cache.k), dev(cache.v), out, dev(positions), dev(torch.zeros(2, dtype=torch.int32)),
                         dev(cache.table), heads, kv_heads, hd, 1.0 / math.sqrt(hd), 0)
    want = cache.values[0][far].double().repeat_interleave(heads // kv_heads, dim=0).reshape(-1)
    for row in out.cpu().double():
        assert float((row - want).abs().max()) < (1e-5 if dtype == torch.float32 else 2e-2)
    if dtype == torch.bfloat16:
        out2 = torch.zeros_like(out)
        es, fp = dev(torch.tensor([0, 2], dtype=torch.int32)), dev(torch.tensor([n - 2], dtype=torch.int32))
        kernels.attn_bf16_prefill(dev(q), dev(cache.k), dev(cache.v), out2, dev(torch.tensor([0, 0], dtype=torch.int32)),
                                  es, fp, dev(cache.table), heads, kv_heads, hd, 1.0 / math.sqrt(hd), 0)
        for row in out2.cpu().double():
            assert float((row - want).abs().max()) < 2e-2


@pytest.mark.parametrize("m,n,k", [(1, 48, 64), (7, 300, 96), (8, 3584, 512), (16, 200, 1544), (17, 331, 520), (33, 1000, 264),
                                   (64, 520, 1024), (48, 130, 72), (64, 4608, 3584),
                                   # past 64 tokens K is walked in chunks of 128: K with a rest, K shorter than a chunk
                                   (65, 331, 520), (80, 1000, 264), (97, 200, 1544), (128, 3584, 1024), (113, 130, 72),
                                   # weight rows a multiple of 4 KB apart: the workgroups start at different chunks
                                   (8, 1100, 2048), (40, 2100, 4096), (100, 1100, 2048)])
@pytest.mark.parametrize("ranges,rows_per_wave", [(1, 1), (1, 2), (3, 1), (8, 2), (2, 110), (1, 114), (3, 109)])
def test_gemm_mid_against_float64(m, n, k, ranges, rows_per_wave):
    from vipera_rs_amd.ops import kernels
    g = torch.Generator().manual_seed(m * 1000 + n + k)
    a = torch.randn(m, k, generator=g).to(torch.bfloat16).to(DEV)
    w = torch.randn(n, k, generator=g).to(torch.bfloat16).to(DEV)
    bias = torch.randn(n, generator=g).to(DEV)
    want = a.double() @ w.double().T + bias.double()
    for out_dtype, tol in ((torch.float32, 1e-5), (torch.bfloat16, 6e-3)):
        out = torch.full((m, n), 7.0, dtype=out_dtype, device=DEV)
        kernels.gemm_bf16_mid(a, w, bias, out, ranges=ranges, rows_per_wave=rows_per_wave)
        assert _rel(out, want) < tol
    base = torch.randn(m, n, generator=g).to(DEV)
    acc = base.clone()
    kernels.gemm_bf16_mid(a, w, None, acc, accumulate=True, ranges=ranges, rows_per_wave=rows_per_wave)
    assert _rel(acc, base.double() + a.double() @ w.double().T) < 1e-5


@pytest.mark.parametrize("m,width,k_in,inter", [(8, 3584, 512, 18944), (1, 256, 64, 32), (16, 512, 1024, 16 * 1000),
                                               (5, 768, 264, 16 * 41), (3, 1024, 3584, 16 * 300), (8, 896, 512, 4864)])
def test_the_norm_split_between_the_products_around_it(m, width, k_in, inter):
    """x += a Wo^T, h = rms_norm(x) * g, out = up(h) * silu(gate(h)) as two kernels: the first also leaves
    bfloat16(x * g) and its workgroups' sums of squares, the second adds those and divides gate and up by the
    root mean square.  Against 64-bit, and against residual product, norm kernel and gated product."""
    from vipera_rs_amd.ops import kernels
    from vipera_rs_amd.ops.linear import interleave_gate_up
    g = torch.Generator().manual_seed(m + width + k_in)
    a = torch.randn(m, k_in, generator=g).to(torch.bfloat16).to(DEV)
    w_o = (torch.randn(width, k_in, generator=g) / k_in ** 0.5).to(torch.bfloat16).to(DEV)
    x0 = (torch.randn(m, width, generator=g) * 2).to(DEV)
    x0[0, 0] = 60.0                                          # one row with a far larger mean square
    gain = (1 + 0.2 * torch.randn(width, generator=g)).to(DEV)
    gate = (torch.randn(inter, width, generator=g) / width ** 0.5).to(torch.bfloat16).to(DEV)
    up = (torch.randn(inter, width, generator=g) / width ** 0.5).to(torch.bfloat16).to(DEV)
    fused = interleave_gate_up(gate, up)
    eps = 1e-5
    x = x0.clone()
    scaled = torch.empty(m, width, dtype=torch.bfloat16, device=DEV)
    sumsq = torch.full((kernels.follow_sumsq_floats(width, m),), 7.0, device=DEV)
    groups = kernels.gemm_bf16_follow(a, w_o, None, x, gain, scaled, sumsq)
    want_x = x0.double() + a.double() @ w_o.double().T
    assert _rel(x, want_x) < 1e-5
    assert _rel(scaled, want_x * gain.double()) < 6e-3
    squares = sumsq[: groups * 16].view(groups, 16).double().sum(0)[:m]
    assert _rel(squares, (want_x ** 2).sum(-1)) < 1e-5
    out = torch.full((m, inter), 7.0, dtype=torch.bfloat16, device=DEV)
    kernels.gemm_bf16_gated_scaled(scaled, fused, out, sumsq, groups, eps)
    h = want_x * torch.rsqrt((want_x ** 2).mean(-1, keepdim=True) + eps) * gain.double()
    gd, ud = h @ gate.double().T, h @ up.double().T
    want = ud * (gd / (1 + torch.exp(-gd)))
    assert _rel(out, want) < 1.2e-2
    # the three kernels it replaces
    x3 = x0.clone()
    kernels.gemm_bf16(a, w_o, None, x3, accumulate=True)
    assert torch.equal(x3, x)
    h3 = torch.empty(m, width, dtype=torch.bfloat16, device=DEV)
    kernels.rmsnorm(x3, gain, eps, h3)
    out3 = torch.empty(m, inter, dtype=torch.bfloat16, device=DEV)
    kernels.gemm_bf16_gated(h3, fused, out3, 0)
    assert _rel(out, out3.double()) < 1.2e-2


@pytest.mark.parametrize("tiling", [-1, 0, 2, 3, 4, 9, 7, 8, 5, 10, 11, 12])
@pytest.mark.parametrize("m,width,k_in,inter", [(64, 520, 1024, 16 * 21), (33, 1032, 1536, 16 * 40), (17, 264, 2048, 16 * 9),
                                               (300, 3584, 512, 16 * 64), (5, 200, 0, 16 * 30)])
def test_the_tiled_gated_product_divides_by_the_norm_before_it(tiling, m, width, k_in, inter):
    """17 to 64 tokens: the residual product whose K is split over workgroups leaves bfloat16(x * g) and the sums of
    squares (the kernel that adds its ranges does), and the tiled gated product divides gate and up by the root
    mean square.  Every tiling of both tiled kernels; sums of squares made by hand too (k_in 0), for token counts
    and group counts that no product before the norm produces.  Against 64-bit, as the kernels it replaces."""
    from vipera_rs_amd.ops import kernels
    from vipera_rs_amd.ops.linear import interleave_gate_up
    g = torch.Generator().manual_seed(m + width + k_in)
    gain = (1 + 0.2 * torch.randn(width, generator=g)).to(DEV)
    gate = (torch.randn(inter, width, generator=g) / width ** 0.5).to(torch.bfloat16).to(DEV)
    up = (torch.randn(inter, width, generator=g) / width ** 0.5).to(torch.bfloat16).to(DEV)
    fused = interleave_gate_up(gate, up)
    eps = 1e-5
    stride = kernels.follow_stride(m)
    x0 = (torch.randn(m, width, generator=g) * 2).to(DEV)
    x0[m // 2, 3] = 60.0                                      # one row with a far larger mean square
    if k_in and m <= 64:
        a = torch.randn(m, k_in, generator=g).to(torch.bfloat16).to(DEV)
        w_o = (torch.randn(width, k_in, generator=g) / k_in ** 0.5).to(torch.bfloat16).to(DEV)
        x = x0.clone()
        scaled = torch.full((m, width), 7.0, dtype=torch.bfloat16, device=DEV)
        sumsq = torch.full((kernels.follow_sumsq_floats(width, m),), 7.0, device=DEV)
        groups = kernels.gemm_bf16_mid_follow(a, w_o, None, x, 2, 1, gain, scaled, sumsq)
        want_x = x0.double() + a.double() @ w_o.double().T
        assert _rel(x, want_x) < 1e-5
    else:  # 37 groups of uneven shares of each row's squares
        x, want_x = x0, x0.double()
        scaled = (x0 * gain).to(torch.bfloat16)
        groups = 37
        shares = torch.rand(groups, m, generator=g).to(DEV).double() + 0.1
        shares = shares / shares.sum(0, keepdim=True) * (want_x ** 2).sum(-1)
        sumsq = torch.full((groups * stride,), 7.0, device=DEV)
        sumsq.view(groups, stride)[:, :m] = shares.float()
    try:
        kernels.gemm_bf16_force_tiling(tiling)
        act = torch.full((m, inter), 7.0, dtype=torch.bfloat16, device=DEV)
        kernels.gemm_bf16_gated_tile_scaled(scaled, fused, act, sumsq, groups, eps)
        h = want_x * torch.rsqrt((want_x ** 2).mean(-1, keepdim=True) + eps) * gain.double()
        gd, ud = h @ gate.double().T, h @ up.double().T
        want = ud * (gd / (1 + torch.exp(-gd)))
        assert _rel(act, want) < 1.2e-2
        h3 = torch.empty(m, width, dtype=torch.bfloat16, device=DEV)       # the two kernels it replaces are as far
        kernels.rmsnorm(x, gain, eps, h3)                                  # from the 64-bit result, each on its side
        act3 = torch.empty_like(act)
        kernels.gemm_bf16_gated(h3, fused, act3, 3)
        assert _rel(act3, want) < 1.2e-2 and _rel(act, act3.double()) < 2.4e-2
    finally:
        kernels.gemm_bf16_force_tiling(-1)


@pytest.mark.parametrize("m,inter,k", [(1, 32, 64), (5, 48, 96), (8, 18944, 512), (16, 176, 200), (33, 128, 264), (64, 1024, 256),
                                       (65, 64, 72), (300, 208, 136), (2048, 512, 128), (2048, 8208, 72), (100, 4608, 64),
                                       # the resident kernel: one pair on four waves, fewer units than waves, runs of
                                       # uneven length, a wave's stretch inside one pair, many pairs per workgroup
                                       (1, 16, 256), (3, 48, 256), (16, 16 * 37, 512), (5, 16 * 1000, 1024), (8, 16 * 257, 3584),
                                       (16, 16 * 300, 4352), (2, 16 * 4111, 768), (7, 32, 2048),
                                       # weight rows a multiple of 4 KB apart (the LDS-shared kernel's workgroups
                                       # start at different chunks)
                                       (6, 16 * 70, 2048), (40, 16 * 70, 4096),
                                       # 256 does not divide K: the resident kernel walks chunks of 128
                                       (8, 4864, 896), (3, 48, 128), (16, 16 * 37, 384)])
def test_gated_product_and_interleaved_swiglu(m, inter, k):
    from vipera_rs_amd.ops import kernels
    from vipera_rs_amd.ops.linear import gated_resident_fits, interleave_gate_up, linear_gated
    g = torch.Generator().manual_seed(m + inter + k)
    a = torch.randn(m, k, generator=g).to(torch.bfloat16).to(DEV)
    gate = torch.randn(inter, k, generator=g).to(torch.bfloat16).to(DEV)
    up = torch.randn(inter, k, generator=g).to(torch.bfloat16).to(DEV)
    gd, ud = a.double() @ gate.double().T, a.double() @ up.double().T
    want = ud * (gd / (1 + torch.exp(-gd)))
    fused = interleave_gate_up(gate, up)
    assert torch.equal(fused[:16], gate[:16]) and torch.equal(fused[16:32], up[:16])
    for rows_per_wave in (1, 2, 3):
        out = torch.full((m, inter), 7.0, dtype=torch.bfloat16, device=DEV)
        kernels.gemm_bf16_gated(a, fused, out, rows_per_wave)
        assert _rel(out, want) < 8e-3, f"fused epilogue, plan {rows_per_wave}"
    if gated_resident_fits(m, 2 * inter, k):
        out = torch.full((m, inter), 7.0, dtype=torch.bfloat16, device=DEV)
        kernels.gemm_bf16_gated(a, fused, out, 0)
        assert _rel(out, want) < 8e-3, "resident activations"
    out = torch.empty(m, inter, dtype=torch.bfloat16, device=DEV)
    linear_gated(a, fused, out, True)                       # whichever path the dispatch takes
    assert _rel(out, want) < 1.2e-2
    plain = torch.empty(m, inter, dtype=torch.bfloat16, device=DEV)
    linear_gated(a, torch.cat([gate, up]).contiguous(), plain, False)
    assert _rel(plain, want) < 1.2e-2


@pytest.mark.parametrize("count", [1, 3, 4, 1023, 70_000])
def test_a_steps_words_are_fetched_from_pinned_host_memory(count):
    """The kernel that stands for the host-to-device copy of a step's metadata: the words arrive as they are, in
    stream order, also when the pinned buffer is written again after the stream has been drained."""
    from vipera_rs_amd.errors import InvalidArgumentError
    from vipera_rs_amd.ops import kernels
    g = torch.Generator().manual_seed(count)
    host = torch.randint(-2 ** 31, 2 ** 31 - 1, (count,), generator=g, dtype=torch.int64).to(torch.int32).pin_memory()
    out = torch.full((count,), 7, dtype=torch.int32, device=DEV)
    if not kernels.fetch_words(host, out):
        pytest.skip("this runtime gives pinned host memory no device address")
    assert torch.equal(out.cpu(), host)
    torch.cuda.synchronize()
    host.numpy()[:] = 5
    assert kernels.fetch_words(host, out)
    assert int(out.min()) == 5 and int(out.max()) == 5
    with pytest.raises(InvalidArgumentError):
        kernels.fetch_words(torch.zeros(count, dtype=torch.int32), out)   # pageable memory is refused on the host


@pytest.mark.parametrize("heads,kv_heads,hd", [(3, 1, 16), (4, 2, 80), (2, 2, 128), (120, 60, 16)])
@pytest.mark.parametrize("bs", [4, 20, 64, 192])
@pytest.mark.parametrize("window,keep", [(0, 0), (70, 0), (40, 5), (30, 130), (-48, 0)])
def test_32_bit_prompt_attention_at_the_edges_of_its_tiles(heads, kv_heads, hd, bs, window, keep):
    """Portions of 15 to 65 tokens that begin on both sides of a tile of 64 positions, pages that divide a tile, do not, or
    hold several; windows that have given pages back (what those and the free slots hold is NaN), first positions that stay
    visible, a sink, a cap, a bias by distance and a gate; few heads (16 tokens a workgroup) and many (32).  The general kernel
    sums a score in the same order and the softmax over other tiles: 2e-6 as in the tests of both against 64 bits."""
    from types import SimpleNamespace
    from vipera_rs_amd.ops import kernels
    entries = [(15, 15), (80, 17), (129, 65), (263, 16)]
    counts, first = [n for _, n in entries], [kv - n for kv, n in entries]
    cache = _Paged([kv for kv, _ in entries], kv_heads, hd, bs, torch.float32, heads * 7 + bs, stale_nan=True)
    table = cache.table
    if window:
        lowest = [max(0, f + 1 - window) if window > 0 else f - f % -window for f in first]
        table = cache.with_pages_given_back(lowest)
        kept = min((keep + bs - 1) // bs, table.shape[1])
        table[:, :kept] = cache.table[:, :kept]
    starts = [sum(counts[:e]) for e in range(len(counts) + 1)]
    T = starts[-1]
    g = torch.Generator().manual_seed(hd + bs)
    qkv = torch.randn(T, (heads + 2 * kv_heads) * hd, generator=g).to(DEV)
    ints = lambda v: torch.tensor(v, dtype=torch.int32, device=DEV)  # noqa: E731
    positions, entry_of = ints([f + i for f, n in zip(first, counts) for i in range(n)]), ints([e for e, n in enumerate(counts) for _ in range(n)])
    tiles = ints([x for e, n in enumerate(counts) for off in range(0, n, 64) for x in (e, off)])
    k, v, table = cache.k.to(DEV), cache.v.to(DEV), table.to(DEV)
    plain = SimpleNamespace(sink=None, rel=None, keep_first=keep, gate=None)
    full = SimpleNamespace(sink=torch.randn(heads, generator=g).to(DEV), rel=torch.randn(heads, 90, generator=g).to(DEV), keep_first=keep,
                           gate=torch.randn(T, heads, generator=g).to(DEV))
    for extras, cap in ((plain, 0.0), (full, 5.0)):
        want, got = torch.zeros(T, heads * hd, device=DEV), torch.full((T, heads * hd), float("nan"), device=DEV)
        kernels.attn_generic(qkv, k, v, want, positions, entry_of, table, heads, kv_heads, hd, hd ** -0.5, window, softcap=cap, extras=extras)
        kernels.attn_prefill_f32(qkv, k, v, got, tiles, 64, ints(starts), ints(first), table, heads, kv_heads, hd, hd ** -0.5, window,
                                 softcap=cap, extras=extras)
        assert _rel(got.cpu(), want.cpu().double()) < 2e-6


@pytest.mark.parametrize("rows,width", [(3, 64), (37, 132), (5, 1028), (9, 4100)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_passes_over_rows_in_fours_give_the_bits_of_one_number_at_a_time(rows, width, dtype):
    """activation, swiglu, head_unpack_gate and scan_prepare where every row lies in pieces of four numbers, against the same
    numbers in rows that do not (an odd stride or an odd width)."""
    from vipera_rs_amd.ops import kernels
    g = torch.Generator(DEV).manual_seed(width)
    randn = lambda *shape: torch.randn(*shape, generator=g, device=DEV)
    odd = lambda x, spare=1: torch.cat([x, x[:, :spare]], dim=1)[:, :x.shape[1]]      # a view of rows one number longer
    x, factor = randn(rows, width).to(dtype), randn(rows, width)
    for kind in kernels.ACTIVATIONS:
        for mul in (None, factor):
            out, apart = torch.empty(rows, width, dtype=dtype, device=DEV), torch.empty(rows, width, dtype=dtype, device=DEV)
            kernels.activation(x, kind, out, mul)
            kernels.activation(odd(x), kind, apart, mul)
            assert torch.equal(out, apart)
    both, pairs = randn(rows, 2 * width).to(dtype), torch.empty(rows, width, dtype=dtype, device=DEV)
    kernels.swiglu(both, pairs)
    lone = torch.empty(rows, width + 1, dtype=dtype, device=DEV)
    kernels.swiglu(torch.cat([odd(both[:, :width + 1])[:, :width], both[:, :1], both[:, width:], both[:, :1]], dim=1).contiguous(), lone)
    assert torch.equal(pairs, lone[:, :width])
    heads = randn(rows, 2 * width).to(dtype)                    # two heads of width - 4 in width columns each
    gate, n = randn(rows, 2 * (width - 4)), width - 4
    out, apart = (torch.empty(rows, 2 * n, dtype=dtype, device=DEV) for _ in range(2))
    kernels.head_unpack_gate(heads, gate, "sigmoid", 2, n, width, out)
    kernels.head_unpack_gate(heads, odd(gate), "sigmoid", 2, n, width, apart)
    assert torch.equal(out, apart)
    step, bias, z = randn(rows, width), randn(width), randn(rows, width)
    ones, gates, alone = odd(step), torch.empty(rows, width, device=DEV), torch.empty(rows, width, device=DEV)
    kernels.scan_prepare(ones, bias, odd(z), alone)
    kernels.scan_prepare(step, bias, z, gates)
    assert torch.equal(step, ones) and torch.equal(gates, alone)


@pytest.mark.parametrize("rows,width", [(6143, 64), (6144, 64), (2979, 132), (97, 4100)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_passes_over_many_rows_in_fours_give_the_bits_of_one_number_at_a_time(rows, width, dtype):
    """On both sides of the number from which a thread takes four, 393,216 of them."""
    test_passes_over_rows_in_fours_give_the_bits_of_one_number_at_a_time(rows, width, dtype)


@pytest.mark.parametrize("tokens,channels", [(1, 1), (7, 512), (1100, 508), (1023, 512), (1024, 512), (130, 4100), (997, 4001), (1049, 4001), (8300, 508)])
def test_every_form_of_the_scans_preparation_gives_the_same_bits(tokens, channels):
    """On both sides of the lines between a thread a number and four a thread, in rows on 16 bytes and off them: the bits of steps of
    one token, and 64-bit."""
    from vipera_rs_amd.ops import kernels
    g = torch.Generator(DEV).manual_seed(tokens + channels)
    wide, bias = torch.randn(tokens, 2 * channels + 4, generator=g, device=DEV) * 4, torch.randn(channels, generator=g, device=DEV)
    for step, z in ((wide[:, :channels].clone(), wide[:, -channels:]), (wide.clone()[:, 1:channels + 1], wide[:, 1:channels + 1])):
        first, gate = step.clone(), torch.full((tokens, channels), float("nan"), device=DEV)
        kernels.scan_prepare(step, bias, z, gate)
        assert _rel(step, torch.nn.functional.softplus(first.double() + bias.double())) < 2e-6
        assert _rel(gate, torch.nn.functional.silu(z.double())) < 2e-6
        for t in {0, tokens // 2, tokens - 1}:
            one, alone = first[t:t + 1].clone(), torch.empty(1, channels, device=DEV)
            kernels.scan_prepare(one, bias, z[t:t + 1], alone)
            assert torch.equal(one, step[t:t + 1]) and torch.equal(alone, gate[t:t + 1])


@pytest.mark.parametrize("tokens,width,dtype", [(514, 36, torch.bfloat16), (515, 1028, torch.float32), (640, 64, torch.bfloat16)])
def test_token_shift_in_runs_of_four_gives_the_bits_of_single_tokens(tokens, width, dtype):
    """A step of 512 tokens or more against the same tokens in smaller steps: entries that begin inside a run, behind a state and at
    position 0."""
    from vipera_rs_amd.ops import kernels
    g = torch.Generator(DEV).manual_seed(tokens)
    h, mu = torch.randn(tokens, width, generator=g, device=DEV).to(dtype), torch.randn(3, width, generator=g, device=DEV)
    saved = torch.randn(5, width + 8, generator=g, device=DEV)
    i32 = lambda a: torch.tensor(list(a), dtype=torch.int32, device=DEV)
    starts, first, slots = [0, 201, 202, 205, tokens], [0, 7, 0, 3], [4, 0, 2, 1]
    whole, parts, left = torch.empty(3, tokens, width, dtype=dtype, device=DEV), torch.empty(3, tokens, width, dtype=dtype, device=DEV), saved.clone()
    entry = lambda pieces: i32(i for i, (lo, hi) in enumerate(pieces) for _ in range(lo, hi))
    all_of = list(zip(starts[:-1], starts[1:]))
    kernels.token_shift(h, mu, left, 4, entry(all_of), i32(starts), i32(first), i32(slots), whole, 4)
    one = saved.clone()
    for e, (lo, hi) in enumerate(all_of):
        for at in range(lo, hi, 150):
            end = min(at + 150, hi)
            piece = torch.empty(3, end - at, width, dtype=dtype, device=DEV)
            kernels.token_shift(h[at:end].contiguous(), mu, one, 4, i32([0] * (end - at)), i32([0, end - at]), i32([first[e] + at - lo]), i32([slots[e]]),
                                piece, 1)
            parts[:, at:end] = piece
    assert torch.equal(whole, parts) and torch.equal(left, one)


@pytest.mark.parametrize("tokens,width,dtype", [(515, 256, torch.float32), (515, 260, torch.bfloat16), (2047, 256, torch.bfloat16),
                                                (2049, 256, torch.float32), (4099, 128, torch.bfloat16)])
def test_token_shift_of_narrow_rows_gives_the_bits_of_single_tokens(tokens, width, dtype):
    """On both sides of a row's turn of a workgroup and of the 524,288 numbers from which narrower rows go in runs."""
    test_token_shift_in_runs_of_four_gives_the_bits_of_single_tokens(tokens, width, dtype)


@pytest.mark.parametrize("tokens,heads,k,n", [(1, 2, 64, 64), (64, 3, 128, 192), (65, 2, 192, 100), (200, 1, 320, 33)])
def test_products_per_head_in_tiles_of_64_give_the_bits_of_the_wide_ones(tokens, heads, k, n):
    """K in whole steps of 64 against the same numbers with eight zeros more, which take the tiles of 128 x 128: tokens and outputs that
    end inside a tile, one step and several, gated, outputs on 8 bytes and not."""
    from vipera_rs_amd.ops import kernels
    g = torch.Generator(DEV).manual_seed(tokens + k)
    a, w = torch.randn(tokens, heads, k, generator=g, device=DEV).bfloat16(), torch.randn(heads, n, k, generator=g, device=DEV).bfloat16()
    gate = torch.randn(tokens, heads, generator=g, device=DEV)
    pad = lambda x: torch.nn.functional.pad(x, (0, 8)).contiguous()
    for opened in (None, gate):
        for spare in (0, 5):
            out = [torch.full((tokens, heads * (n + spare)), 7.0, device=DEV).bfloat16() for _ in range(2)]
            kernels.head_linear(a.reshape(tokens, -1), k, k, w, out[0], n + spare, gate=opened)
            kernels.head_linear(pad(a).reshape(tokens, -1), k + 8, k + 8, pad(w), out[1], n + spare, gate=opened)
            assert torch.equal(out[0], out[1])
    want = torch.einsum("thk,hnk->thn", a.double().cpu(), w.double().cpu()) * torch.sigmoid(gate.double().cpu())[..., None]
    got = out[0].reshape(tokens, heads, n + 5)[..., :n].double().cpu()
    assert float((got - want).abs().max()) <= 2.0 ** -8 * float(want.abs().max())      # outputs are rounded to bfloat16


@pytest.mark.parametrize("tokens", [5, 70])
@pytest.mark.parametrize("experts,top", [(1, 1), (5, 4), (33, 4), (64, 6), (130, 4)])
def test_routes_by_lane_moves_are_the_largest_logits_lowest_id_first(tokens, experts, top):
    """A token's choices over one and several experts a lane, whole numbers so that many are equal, and the grouping by expert: the
    counts, the places and the tiles as a sort in plain code gives them."""
    from vipera_rs_amd.ops import kernels
    g = torch.Generator().manual_seed(experts + tokens)
    logits = torch.randint(-3, 4, (tokens, experts), generator=g).float()
    logits[torch.rand(tokens, experts, generator=g) < 0.1] = float("-inf")
    i32 = lambda n: torch.full((n,), -7, dtype=torch.int32, device=DEV)
    pairs = tokens * top
    ids, offsets, order, tiles, count = i32(pairs), i32(experts + 1), i32(pairs), i32(2 * kernels.moe_max_tiles(pairs, experts, 64)), i32(1)
    weights = torch.empty(pairs, device=DEV)
    kernels.moe_route(logits.to(DEV), top, ids, weights, offsets, order, tiles, count)
    want = [sorted(range(experts), key=lambda e: (-logits[t, e].item(), e))[:top] for t in range(tokens)]
    assert ids.cpu().view(tokens, top).tolist() == want
    flat = [e for row in want for e in row]
    starts = [sum(x < e for x in flat) for e in range(experts + 1)]
    assert offsets.tolist() == starts
    placed = order.tolist()
    assert sorted(placed) == list(range(pairs)) and all(flat[p] == e for e in range(experts) for p in placed[starts[e]:starts[e + 1]])
    assert tiles.tolist()[:2 * count.item()] == [x for e in range(experts) for first in range(starts[e], starts[e + 1], 64) for x in (e, first)]


# every form of the 32-bit product, at sizes with remainders of its tiles, and one of several slabs in each form that walks them
@pytest.mark.parametrize("m,inter,k", [
    (9, 4, 132), (17, 20, 896), (17, 2404, 896), (130, 1004, 896), (333, 516, 1024), (700, 4868, 1024), (50, 4868, 64), (50, 4864, 132),
    (17, 8968, 260), (65, 4868, 1536), (333, 4864, 132), (333, 2404, 1028), (333, 2404, 896), (65, 8962, 896), (130, 2405, 896)])
def test_gated_32_bit_product_has_the_bits_of_product_and_gate(m, inter, k):
    from vipera_rs_amd.ops import kernels

    gen = torch.Generator("cuda").manual_seed(m + inter + k)
    a = torch.randn(m, k, generator=gen, device="cuda")
    w = torch.randn(2 * inter, k, generator=gen, device="cuda") * k ** -0.5
    a[0, 0] = 1e30     # a row of gates far out on both sides
    both, want = torch.empty(m, 2 * inter, device="cuda"), torch.empty(m, inter, device="cuda")
    kernels.gemm_generic(a, w, None, both)
    kernels.swiglu(both, want)
    got = torch.full((m, inter), float("nan"), device="cuda")
    assert kernels.gemm_generic_gated(a, w, got)
    assert torch.equal(got, want)
    strided = torch.empty(m, k + 4, device="cuda")
    strided[:, :k] = a
    assert kernels.gemm_generic_gated(strided[:, :k], w, got.fill_(0.0)) and torch.equal(got, want)


def test_gated_32_bit_product_leaves_what_it_cannot_take():
    from vipera_rs_amd.ops import kernels

    a, w, out = torch.ones(65, 1028, device="cuda"), torch.ones(24, 1028, device="cuda"), torch.zeros(65, 12, device="cuda")
    assert not kernels.gemm_generic_gated(a, w, out)                                   # parts of its sums in memory
    assert not kernels.gemm_generic_gated(a[:8, :64], w[:, :64].contiguous(), out[:8])      # a stream of the weights
    room = torch.ones(65 * 64 + 1, device="cuda")
    assert not kernels.gemm_generic_gated(room[1:].view(65, 64), w[:, :64].contiguous(), out)     # rows off 16 bytes
    assert not out.any()


def test_gated_32_bit_layer_may_write_over_its_input():
    from vipera_rs_amd.ops import kernels
    from vipera_rs_amd.ops.linear import linear_gated

    gen = torch.Generator("cuda").manual_seed(8)
    m, k = 130, 896
    room, w = torch.randn(2 * m, k, generator=gen, device="cuda"), torch.randn(2 * k, k, generator=gen, device="cuda") * k ** -0.5
    for at in (0, 7, 129, 130):                # the input's own rows, rows that overlap with them, and the next ones
        a = room.clone()[:m]
        out = a.as_strided((m, k), (k, 1), at * k)
        assert kernels.gemm_generic_gated(a, w, torch.empty_like(a))
        want = torch.empty_like(a)
        linear_gated(a, w, want, False)
        if at < m:
            assert not kernels.gemm_generic_gated(a, w, out)
        linear_gated(a, w, out, False)
        assert torch.equal(out, want)
