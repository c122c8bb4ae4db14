"""64-row tiles (weights decoded straight into MFMA operands, activations through LDS in four-stage chunks) against the
256-row kernel (weights decoded through LDS) bit for bit, and against the CPU oracle: row counts around every 16-row
group, K of whole and partial chunks, every trellis width."""
import numpy as np
import pytest
import torch

import exl3_grouped as gp
import exl3_oracle as O
from exl3_grouped import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bits", [2, 3, 4])
@pytest.mark.parametrize("K", [64, 128, 192, 320, 768])       # 2, 4, 6, 10 and 24 stages
def test_thin_tiles_match_256_row_tiles(dev, bits, K):
    N = 256
    a, packed, svh = synth.make_fat(bits * 1000 + K, M=64, K=K, N=N, bits=bits)
    ref = O.fat_gemm(a, packed, svh, dtype=np.float64)
    ta, tp, ts = (torch.from_numpy(v).to(dev) for v in (a, packed, svh))
    for m in (1, 15, 16, 17, 31, 32, 33, 47, 48, 49, 63, 64):
        got = {}
        for variant in (0, 2):                                 # 64-row tiles, 256-row tiles
            out = torch.full((m, N), float("nan"), dtype=torch.float32, device=dev)
            gp.fat_gemm_v2(ta[:m], tp, out, ts, bits, True, False, variant)
            got[variant] = out.cpu().numpy()
        assert np.array_equal(got[0].view(np.uint32), got[2].view(np.uint32)), m
        # fp16 products are exact in fp32: what is left is the rounding of K + 128 fp32 sums per output, 2^-24 each and
        # random in sign, so sqrt(K + 128) 2^-24 <= 1.8e-6 in the 2-norm
        assert O.rel_l2(got[0], ref[:m]) < 2e-6, m
