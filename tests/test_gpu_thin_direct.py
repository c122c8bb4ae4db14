"""64- and 128-row tiles (weights decoded straight into MFMA operands, activations through LDS in four-stage chunks) against the
256-row kernel (weights decoded through LDS) bit for bit, and against the CPU oracle: row counts around every 16-row
group, K of whole and partial chunks, every trellis width."""
import ctypes

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


@pytest.mark.parametrize("bits", [2, 3, 4])
@pytest.mark.parametrize("K", [64, 192, 768])
def test_grouped_128_row_tiles_match_256_row_tiles(dev, bits, K):
    """One tile per expert, row counts around every 16-row group up to 128: fp16 T16 rows of two tensors, per-route fp32
    rows and the atomic scatter (one add per token) on a 128-row table against a 256-row one."""
    rows = [128, 1, 16, 17, 64, 65, 80, 81, 96, 97, 112, 113, 127]
    E, N, R = len(rows), 256, sum(rows)
    rng = np.random.default_rng(bits * 100 + K)
    words = torch.from_numpy(rng.integers(-32768, 32768, (E, 2, K // 16, N // 16, 16 * bits), dtype=np.int16)).to(dev)
    svh = torch.from_numpy((rng.uniform(0.5, 1.5, (E, 2, N))).astype(np.float16)).to(dev)
    a = torch.from_numpy(rng.standard_normal((gp.t16_rows(R), K)).astype(np.float16)).to(dev)
    counts = torch.tensor(rows, dtype=torch.int32, device=dev)
    row0 = (torch.cumsum(counts, 0) - counts).to(torch.int32)
    experts = torch.arange(E, dtype=torch.int32, device=dev)
    rw = torch.from_numpy(rng.uniform(0.1, 1, R).astype(np.float16)).to(dev)
    route = torch.from_numpy(rng.permutation(R).astype(np.int32)).to(dev)
    got = {}
    for tr in (128, 256):
        kw = dict(tile_rows=tr, a_layout=1, a_rows=R, weights_once=tr == 128)
        gu = torch.full((gp.t16_rows(R), 2 * N), float("nan"), dtype=torch.float16, device=dev)
        gp.grouped_gemm(a, words[:, 0], words[:, 1], svh[:, 0], svh[:, 1], experts, row0, counts, row0, None, None, gu, 4,
                        **kw)
        per_route = torch.full((R, N), float("nan"), dtype=torch.float32, device=dev)
        gp.grouped_gemm(a, words[:, 0], None, svh[:, 0], None, experts, row0, counts, row0, None, rw, per_route, 2,
                        route_index=route, **kw)
        out = torch.zeros(R, N, dtype=torch.float32, device=dev)
        gp.grouped_gemm(a, words[:, 0], None, svh[:, 0], None, experts, row0, counts, row0, route.long(), rw, out, 1, **kw)
        got[tr] = [t.cpu().numpy() for t in (gu.view(torch.int16), per_route.view(torch.int32), out.view(torch.int32))]
        assert torch.equal(out, per_route)                     # one add onto zero per row
    for x, y in zip(got[128], got[256]):
        assert np.array_equal(x, y)


@pytest.mark.parametrize("tile_rows,thin_rows,T", [(128, 128, 700), (256, 128, 700), (256, 128, 120), (256, 128, 4000),
                                                   (512, 128, 700), (256, 64, 700)])
def test_tail_tables(dev, tile_rows, thin_rows, T):
    """sort_routes_tail_tiles' two tables against a closed form, at the smallest table the bound allows."""
    rng = np.random.default_rng(tile_rows + thin_rows)
    E, k = 24, 4
    p = rng.uniform(0, 1, E) ** (1 if T > 1000 else 3)
    ids = np.stack([rng.choice(E, k, replace=False, p=p / p.sum()) for _ in range(T)])
    R, counts = T * k, np.bincount(ids.ravel(), minlength=E)
    rem = counts % tile_rows
    mid, big = ((rem > 64) & (rem <= 128)).sum(), (counts // tile_rows + (rem > 128)).sum()
    limit = thin_rows if 2 * mid > big else 64
    full, thin, row = [], [], 0
    for e, c in enumerate(counts):
        for r in range(0, c, tile_rows):
            (thin if c - r <= limit and c - r < tile_rows else full).append((e, row + r))
        row += c
    mf, mt = min(R // tile_rows + E, max(1, R // min(tile_rows, 65))), min(E, R)
    assert len(full) <= mf
    i32 = lambda n: torch.full((n,), -7, dtype=torch.int32, device=dev)  # noqa: E731
    fe, fr, te, tr, meta, cnt, row0, eor = i32(mf), i32(mf), i32(mt), i32(mt), i32(3), i32(E), i32(E), i32(R)
    ts, ws = torch.empty(R, dtype=torch.int64, device=dev), torch.empty(R, dtype=torch.float16, device=dev)
    gp.sort_routes_tail_tiles(torch.from_numpy(ids).to(dev), torch.ones(T, k, device=dev), E, ts, ws, eor, cnt, row0, fe, fr,
                              te, tr, meta, tile_rows, thin_rows)
    assert meta.tolist() == [len(full), R, len(thin)] and cnt.tolist() == counts.tolist()
    for tab, e, r in ((full, fe, fr), (thin, te, tr)):
        assert list(zip(e.tolist(), r.tolist()))[:len(tab)] == tab
        assert (e[len(tab):] == -1).all()


def kernels_of(fn):
    """Names of the kernels `fn` launches, from a graph that captures it (nothing runs)."""
    hip = ctypes.CDLL("libamdhip64.so")
    hip.hipKernelNameRefByPtr.restype = ctypes.c_char_p
    graph = torch.cuda.CUDAGraph(keep_graph=True)
    with torch.cuda.graph(graph):
        fn()
    raw, n = ctypes.c_void_p(graph.raw_cuda_graph()), ctypes.c_size_t()
    assert hip.hipGraphGetNodes(raw, None, ctypes.byref(n)) == 0
    nodes = (ctypes.c_void_p * n.value)()
    assert hip.hipGraphGetNodes(raw, nodes, ctypes.byref(n)) == 0

    class Params(ctypes.Structure):                            # hipKernelNodeParams
        _fields_ = [("block", ctypes.c_uint32 * 3), ("extra", ctypes.c_void_p), ("func", ctypes.c_void_p),
                    ("grid", ctypes.c_uint32 * 3), ("params", ctypes.c_void_p), ("shared", ctypes.c_uint32)]
    names = []
    for node in nodes:
        p = Params()
        assert hip.hipGraphKernelNodeGetParams(ctypes.c_void_p(node), ctypes.byref(p)) == 0
        names.append(hip.hipKernelNameRefByPtr(ctypes.c_void_p(p.func), None).decode())
    return names


@pytest.mark.parametrize("tile_rows", [64, 128])
@pytest.mark.parametrize("mode", [0, 1, 2, 4])
def test_weights_are_streamed_only_when_read_once(dev, tile_rows, mode):
    """A table may hold many tiles of an expert, which share its weights through the caches: only weights_once (and not
    with the atomic scatter) takes the kernel with non-temporal weight loads, the last template argument."""
    E, K, N, R = 2, 128, 128, 400
    words = torch.zeros(E, K // 16, N // 16, 64, dtype=torch.int16, device=dev)
    half = lambda *s: torch.ones(*s, dtype=torch.float16, device=dev)  # noqa: E731
    table = torch.zeros(4, dtype=torch.int32, device=dev)
    out = torch.zeros(gp.t16_rows(R), N, dtype=torch.float16 if mode in (0, 4) else torch.float32, device=dev)
    rows = torch.arange(R, dtype=torch.int32, device=dev)
    tokens = rows.long()
    a, svh, rw, counts = half(gp.t16_rows(R), K), half(E, N), half(R), torch.tensor([R, 0], dtype=torch.int32, device=dev)
    for once in (False, True):
        names = kernels_of(lambda: gp.grouped_gemm(
            a, words, None, svh, None, table, table, counts, table[:E], tokens if mode == 1 else None,
            rw if mode in (1, 2) else None, out if mode == 4 else out[:R], mode, route_index=rows if mode == 2 else None,
            tile_rows=tile_rows, a_layout=1, a_rows=R, weights_once=once))
        assert len(names) == 1 and "trellis_gemm_kernelILi4E" in names[0], names
        assert ("Lb1EEE" in names[0]) == (once and mode != 1), names
