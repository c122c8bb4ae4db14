"""bf16 activations read as they are (each value rounded to fp16 inside the input Hadamard) against a cast in front, bit for
bit: the Hadamard pass over ragged row counts and special values, the prefill and decode paths, and rows at an address
the kernels cannot load 16 bytes from, which are cast first."""
import numpy as np
import pytest
import torch

import exl3_grouped as gp
import exl3_grouped_runtime as rt
from exl3_grouped import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", [1, 15, 16, 17, 130])
def test_row_had_gather_bf16(dev, rows):
    K, tokens, E = 384, 40, 5
    g = torch.Generator().manual_seed(rows)
    x = torch.randn(tokens, K, generator=g).to(torch.bfloat16)
    x[0, :8] = torch.tensor([65504.0, 65536.0, 1e-7, 3e-8, -0.0, 6e-5, 3e38, -1e-6]).to(torch.bfloat16)
    x = x.to(dev)
    tok = torch.randint(0, tokens, (rows,), generator=g).to(dev)
    tok[0] = 0
    eor = torch.randint(0, E, (rows,), generator=g).to(torch.int32).to(dev)
    suh = (torch.randint(0, 2, (E, K), generator=g) * 2 - 1).to(torch.float16).to(dev)
    got, ref = (torch.full((gp.t16_rows(rows), K), float("nan"), dtype=torch.float16, device=dev) for _ in range(2))
    gp.row_had_gather_bf16(x, got, tok, eor, suh, rows)
    gp.row_had(x.to(torch.float16), ref, tok, eor, suh, True, dst_layout=1, rows=rows)
    assert torch.equal(got.view(torch.int16), ref.view(torch.int16))


@pytest.mark.parametrize("T,shift", [(1, 0), (5, 0), (5, 1), (40, 0), (40, 1), (128, 0)])
def test_layer_bf16_matches_cast(dev, T, shift):
    L, _, _, _, cfg = synth.make_config("tiny", seed=3)
    TL = synth.to_device(L, dev)
    ids, w = synth.make_routing("softmax", T, cfg["E"], cfg["topk"], 9)
    ids, w = torch.from_numpy(ids).to(dev), torch.from_numpy(w).to(dev)
    flat = torch.randn(T * cfg["H"] + 8, generator=torch.Generator().manual_seed(T)).to(torch.bfloat16).to(dev)
    x = flat[shift:shift + T * cfg["H"]].view(T, cfg["H"])       # shift 1: contiguous, 2 bytes off a 16-byte address
    assert (x.data_ptr() % 16 == 0) == (shift == 0)
    a = rt.grouped_prefill(x, ids, w, TL, 10.0, scatter="combine")
    b = rt.grouped_prefill(x.to(torch.float16), ids, w, TL, 10.0, scatter="combine")
    assert torch.equal(a.view(torch.int32), b.view(torch.int32))
    layer = (TL.w13_trellis, TL.w13_suh, TL.w13_svh, TL.w2_trellis, TL.w2_suh, TL.w2_svh)
    rt._decode_ws.clear()                                       # sized by this test
    got = [rt.moe_decode(x, ids, w, TL, 10.0)]                  # shift 1: cast in front
    if shift == 0:
        got.append(gp.moe_decode_dt(x, ids, w, *layer, 10.0))
    rt._decode_ws.clear()                                       # later tests size their own
    d = gp.moe_decode(x.to(torch.float16), ids, w, *layer, 10.0)
    for c in got:
        # the same launches add fp32 partial sums in an order of their own: a few 2^-24 per sum, and an fp16 step of a
        # gate|up value where that crosses a rounding boundary
        assert (c - d).norm() <= 1e-4 * d.norm()
