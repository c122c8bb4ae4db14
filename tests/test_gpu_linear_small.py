"""The dense linear at few rows (64-row tiles, with four K slices in one workgroup where that pays) against the same
projection through the per-expert GEMM on 256-row tiles: row counts around each 16-row group and past one tile, sliced
and unsliced lengths, every trellis width and both output types; and which sizes are sliced."""
import numpy as np
import pytest
import torch

import exl3_grouped as gp
from exl3_grouped import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bits", [2, 3, 4])
@pytest.mark.parametrize("K,N", [(256, 384), (384, 384), (768, 384), (1280, 384),     # unsliced; unsliced, 10 stages a slice
                                 (2048, 384), (2048, 4096)])                          # fp32: two slices, four slices
def test_linear_few_rows(dev, bits, K, N):
    x, packed, svh = synth.make_fat(bits * 100 + K, M=200, K=K, N=N, bits=bits)
    suh = np.random.default_rng(K).integers(0, 2, K).astype(np.float16) * 2 - 1
    x, packed, svh, suh = (torch.from_numpy(v).to(dev) for v in (x, packed, svh, suh))
    for m in (1, 7, 16, 17, 33, 64, 65, 200):
        h = torch.empty(m, K, dtype=torch.float16, device=dev)
        gp.row_had(x[:m], h, None, torch.zeros(m, dtype=torch.int32, device=dev), suh[None], False)
        ref = torch.empty(m, N, dtype=torch.float32, device=dev)
        gp.fat_gemm_v2(h, packed, ref, svh, bits, True, False, 2)
        y = gp.linear_exl3(x[:m], packed, suh, svh, K=bits, out_dtype=torch.float32)
        # the same exact products, their K + 128 fp32 sums in another order: sqrt(K + 128) 2^-24 for each side
        assert (y - ref).norm() <= 4.5e-6 * ref.norm(), m
        again = gp.linear_exl3(x[:m], packed, suh, svh, K=bits, out_dtype=torch.float32)
        assert torch.equal(y.view(torch.int32), again.view(torch.int32))
        y16 = gp.linear_exl3(x[:m], packed, suh, svh, K=bits)
        # one fp16 rounding of y (2^-11, and the fp32 path's rounded product) and, where the two outputs run different
        # schedules (K = 2048, 3 tiles), the order of K + 128 sums, each rounding a partial sum of the result's size
        order = (K + 128) * 2.0 ** -24 * y.square().mean().sqrt()
        assert (y16.float() - y).abs().le(y.abs() * 2 ** -10.9 + order).all(), m


@pytest.mark.parametrize("m,K,N,f32,sliced", [
    (7, 1024, 4096, True, True), (7, 1024, 4224, True, False),        # 32 and 33 tiles of one row group
    (64, 768, 4096, True, False), (64, 256, 384, False, False),       # a slice of 6 and of 2 stages
    (520, 1024, 2048, True, True), (520, 1024, 2176, True, False),    # 9 row groups: 2 x 16 and 2 x 17 tiles
    (64, 4096, 8192, False, False), (64, 6144, 8192, False, True),    # 64 tiles, two rounds
    (64, 6144, 8320, False, False),                                   # 65 tiles
    (7, 4096, 2048, True, False), (7, 4096, 2176, True, True),        # against the two K slices of the fp32 output
    (7, 6144, 6144, True, False), (7, 2048, 23040, False, False)])    # two rounds; 180 column tiles
def test_linear_schedule_by_size(dev, m, K, N, f32, sliced):
    """Which calls the K-slice schedule takes: it sums four parts of K, so its bits differ from the other schedules', which
    give those of the grouped GEMM's 64-row tiles (fp32 with K >= 2048: of the per-expert GEMM's two K slices)."""
    g = torch.Generator(device=dev).manual_seed(K + N)
    x = torch.randn(m, K, device=dev, generator=g).half()
    packed = torch.randint(-32768, 32768, (K // 16, N // 16, 64), dtype=torch.int16, device=dev, generator=g)
    suh = (torch.randint(0, 2, (K,), device=dev, generator=g) * 2 - 1).half()
    svh = (torch.rand(N, device=dev, generator=g) + 0.5).half()
    dt = torch.float32 if f32 else torch.float16
    zeros = torch.zeros(m, dtype=torch.int32, device=dev)
    h = torch.empty(m, K, dtype=torch.float16, device=dev)
    gp.row_had(x, h, None, zeros, suh[None], False)
    ref = torch.empty(m, N, dtype=dt, device=dev)
    if f32 and K >= 2048:
        gp.fat_gemm_v2(h, packed, ref, svh, 4, True, False)
    else:
        tiles = (m + 63) // 64
        row0 = 64 * torch.arange(tiles, dtype=torch.int32, device=dev)
        one, rows = torch.ones(m, dtype=torch.float16, device=dev), torch.arange(m, dtype=torch.int32, device=dev)
        gp.grouped_gemm(h, packed[None], None, svh[None], None, zeros[:1].expand(tiles).contiguous(), row0,
                        torch.full((1,), m, dtype=torch.int32, device=dev), zeros[:1], None, one if f32 else None, ref,
                        2 if f32 else 0, route_index=rows if f32 else None, tile_rows=64)
    y = gp.linear_exl3(x, packed, suh, svh, out_dtype=dt)
    # K + 128 fp32 sums in another order, 2^-24 sqrt(K + 128) <= 5e-6 for each side; fp16: at most one rounding (2^-11)
    assert (y.float() - ref.float()).norm() <= (1e-5 if f32 else 2 ** -11) * ref.float().norm()
    assert torch.equal(y, ref) == (not sliced)
