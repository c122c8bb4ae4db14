"""The dense linear at few rows (64-row tiles with four K slices in one workgroup where K is a multiple of 256) against the
same projection through the per-expert GEMM on 256-row tiles: row counts around each 16-row group and past one tile,
the shortest and odd slice lengths, every trellis width and both output types."""
import numpy as np
import pytest
import torch

import exl3_grouped as gp
from exl3_grouped import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bits", [2, 3, 4])
@pytest.mark.parametrize("K,N", [(256, 384), (384, 384), (768, 384), (1280, 384),     # 2, unsplit, 6, 10 stages a slice
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
