"""Float32 kernels at the edges of their tiles and loaders: contractions, widths and ranks that
are whole 16-byte chunks (direct-to-LDS loads) and that are not (element loads), grids of every tile
size, several splits of the reductions, pitched operands. Reference: the same products in float64.

Bound: a float32 sum of n products in any order is within n·2^-24 of exact in the worst case and
near sqrt(n)·2^-24 for random signs; at n <= 2052 + 256 that is 2.9e-6 relative to the sum of
magnitudes' rms (4.0e-6 in the reductions over at most 4400 rows), so rel-L2 <= 5e-6 holds, while a dropped
row, column or chunk of a tile (1 of at most 256 terms) changes the result by more than 1e-3.
"""
import pytest
import torch

pytestmark = pytest.mark.gpu
TOL = 5e-6


def rel(got, want):
    return ((got.double() - want).norm() / want.norm().clamp_min(1e-300)).item()


def pitched(t, pad):
    """t as a view of rows that are `pad` elements further apart."""
    if not pad:
        return t
    wide = torch.full((t.shape[0], t.shape[1] + pad), float("nan"), device=t.device)
    wide[:, :t.shape[1]] = t
    return wide[:, :t.shape[1]]


@pytest.mark.parametrize("lengths,ids,K,N,ranks,pad", [
    ((33, 0, 95), (0, 1, -1), 32, 64, (8, 4), 0),                 # one k-tile, 32-row shrink tiles
    ((500, 12), (0, 1), 260, 256, (8, 8), 4),                     # split-contraction tiles, partial k-tile
    ((127, 1, 129, 256), (1, -1, 0, 1), 132, 516, (64, 32), 0),   # split-contraction tiles, column remainder
    ((2049, 1023, 1100), (0, 1, 0), 388, 2052, (128, 256), 8),    # 64x64 tiles, two rank blocks, splits
    ((2049, 1023, 1100), (0, 1, 0), 387, 2050, (128, 255), 0),    # the same sizes off the 16-byte chunks
    ((70, 59), (0, 1), 31, 65, (5, 1), 3),                        # element loads, one k-tile
    ((65, 64), (0, 1), 64, 96, (36, 100), 1),                     # chunks whole, pitch not
    ((2500, 3, 1897, 1900), (0, -1, 1, 0), 2052, 2052, (64, 32), 4),  # 128x64 tiles cut by segments, both products
    ((2500, 3, 1897, 1900), (0, -1, 1, 0), 2050, 2051, (63, 30), 0),  # the same through the element loads
])
def test_f32_kernels_at_tile_edges(pkg, dev, lengths, ids, K, N, ranks, pad):
    k = pkg.kernels
    g = torch.Generator().manual_seed(K + N)
    M = sum(lengths)
    routing = pkg.SegmentRouting.from_lengths(lengths, ids)
    x = pitched(torch.randn(M, K, generator=g).to(dev), pad)
    dy = pitched(torch.randn(M, N, generator=g).to(dev), pad)
    w = pitched((torch.randn(N, K, generator=g) / K ** 0.5).to(dev), pad)
    b = torch.randn(N, generator=g).to(dev)
    As = [(torch.randn(r, K, generator=g) / K ** 0.5).to(dev) for r in ranks]
    Bs = [(torch.randn(N, r, generator=g) * 0.1).to(dev) for r in ranks]
    scales = [0.5, 2.0]
    width = max(ranks)
    h = k.f32_shrink(x, As, 0, scales, routing, width)
    gr = k.f32_shrink(dy, Bs, 1, scales, routing, width)
    y = k.f32_gemm_fwd(x, w, b, h, Bs, routing)
    dx = k.f32_gemm_dx(dy, w, gr, As, routing)
    dB = k.f32_seg_outer(dy, h, ranks, routing, 0)
    dA = k.f32_seg_outer(x, gr, ranks, routing, 1)
    xd, dyd, wd = x.double(), dy.double(), w.double()
    h_ref = torch.zeros(M, width, device=dev, dtype=torch.float64)
    g_ref = torch.zeros_like(h_ref)
    y_ref, dx_ref = xd @ wd.t() + b.double(), dyd @ wd
    dA_ref = [torch.zeros(r, K, device=dev, dtype=torch.float64) for r in ranks]
    dB_ref = [torch.zeros(N, r, device=dev, dtype=torch.float64) for r in ranks]
    r0 = 0
    for n, a in zip(lengths, ids):
        rows = slice(r0, r0 + n)
        r0 += n
        if a < 0 or n == 0:
            continue
        r = ranks[a]
        h_ref[rows, :r] = scales[a] * (xd[rows] @ As[a].double().t())
        g_ref[rows, :r] = scales[a] * (dyd[rows] @ Bs[a].double())
        y_ref[rows] += h_ref[rows, :r] @ Bs[a].double().t()
        dx_ref[rows] += g_ref[rows, :r] @ As[a].double()
        dB_ref[a] += dyd[rows].t() @ h_ref[rows, :r]
        dA_ref[a] += g_ref[rows, :r].t() @ xd[rows]
    assert rel(h, h_ref) <= TOL and rel(gr, g_ref) <= TOL
    assert not h[h_ref == 0].any() and not gr[g_ref == 0].any()  # rows and columns of no adapter
    assert rel(y, y_ref) <= TOL and rel(dx, dx_ref) <= TOL
    for a in range(len(ranks)):
        if dA_ref[a].any():
            assert rel(dA[a], dA_ref[a]) <= TOL and rel(dB[a], dB_ref[a]) <= TOL
        else:
            assert not dA[a].any() and not dB[a].any()


@pytest.mark.parametrize("C,ranks", [(132, (8, 64)), (130, (7, 63)), (260, (256, 0))])
@pytest.mark.parametrize("layout", [0, 1])
def test_reduction_without_a_workspace_is_the_split_one(pkg, dev, C, ranks, layout):
    """mlora_f32_seg_outer (no workspace: every adapter's rows in one run) against the split form and float64;
    an adapter without rows gets zeros."""
    L, lib = pkg._lib, pkg._lib.load()
    g = torch.Generator().manual_seed(C)
    lengths, ids = (700, 33, 0, 1500), (0, -1, 1, 0)
    M, ranks = sum(lengths), (*ranks, 12)
    ids = (0, -1, 2, 1) if ranks[1] else ids
    p, h = torch.randn(M, C, generator=g).to(dev), torch.randn(M, 256, generator=g).to(dev)
    routing = pkg.SegmentRouting.from_lengths(lengths, ids)
    outs = [torch.full((C, r) if layout == 0 else (r, C), float("nan"), device=dev) for r in ranks]
    L.check("mlora_f32_seg_outer", lib.mlora_f32_seg_outer(
        p.data_ptr(), C, M, C, h.data_ptr(), 256, L.ptr_array([o.data_ptr() for o in outs]), layout, L.i32_array(ranks),
        len(ranks), L.i64_array(routing.seg_offsets), L.i32_array(routing.adapter_ids), len(ids),
        torch.cuda.current_stream().cuda_stream))
    split = pkg.kernels.f32_seg_outer(p, h, ranks, routing, layout)
    for a, r in enumerate(ranks):
        want = torch.zeros(C, r, device=dev, dtype=torch.float64)
        for s, ad in enumerate(ids):
            rows = slice(routing.seg_offsets[s], routing.seg_offsets[s + 1])
            if ad == a:
                want += p[rows].double().t() @ h[rows, :r].double()
        want = want if layout == 0 else want.t()
        if want.any():
            assert rel(outs[a], want) <= TOL and rel(split[a], want) <= TOL
        else:
            assert not outs[a].any() and not split[a].any()
