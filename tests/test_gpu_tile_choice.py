"""GEMM tile choice: every output takes its products in the same order in every tile size, so a call
on the first m rows of a batch must give the first m rows of the whole batch's result bit for bit,
whichever tiles the two grids run (64x64, 128x128, 128x256, 256x128, one partly filled round of
256x256, whole rounds and a tail). Row counts sit on both sides of each choice at N = 1544 (a partial
last column tile of every size); the contractions are whole k-tiles, a partial one and shorter than
one; the segment boundaries fall inside tiles. The whole batch is checked against float64 products
on sampled rows (one bf16 rounding: 2e-3)."""
import pytest
import torch

pytestmark = pytest.mark.gpu
N, R = 1544, 72
ROWS = (1, 63, 65, 640, 1153, 1281, 2300, 2500, 4300, 5300, 9300)  # of M = 20500


def _sub(pkg, lengths, ids, m):
    out, left = [], m
    for n in lengths:
        out.append(min(n, left))
        left -= out[-1]
    return pkg.SegmentRouting.from_lengths(out, ids)


@pytest.mark.parametrize("K", [1536, 1000, 40])
def test_rows_do_not_depend_on_the_tile_size(pkg, dev, K):
    k = pkg.kernels
    g = torch.Generator().manual_seed(K)
    M, lengths, ids = 20500, (500, 700, 0, 3000, 5000, 11300), (0, 1, 0, -1, 1, 0)
    rand = lambda *s, std=1.0: (torch.randn(*s, generator=g) * std).to(torch.bfloat16).to(dev)  # noqa: E731
    x, w, b, h = rand(M, K), rand(N, K, std=K ** -0.5), rand(N), rand(M, R, std=0.3)
    bs = [rand(N, R, std=0.05) for _ in range(2)]
    routing = pkg.SegmentRouting.from_lengths(lengths, ids)
    y = k.gemm_fwd(x, w, b, h, bs, routing)
    rows = torch.arange(0, M, 173, device=dev)
    ref = x[rows].double() @ w.double().t() + b.double()
    adapter = torch.tensor(routing.row_adapter(), device=dev)[rows]
    for a in range(2):
        ref += torch.where((adapter == a)[:, None], h[rows].double() @ bs[a].double().t(), 0)
    assert ((y[rows].double() - ref).norm() / ref.norm()).item() <= 2e-3
    wt, ats = w.t().contiguous(), [t.t().contiguous() for t in bs]  # the NN form of the same product
    nn = k.gemm_dx(x, wt, h, ats, routing)
    if K % 16 == 0:
        xq, xs = k.quantize_rows_fp8(x)
        wq, ws = k.quantize_rows_fp8(w)
        y8 = k.gemm_fwd_fp8(xq, xs, wq, ws, b, h, bs, routing)
    for m in ROWS:
        sub = _sub(pkg, lengths, ids, m)
        assert torch.equal(k.gemm_fwd(x[:m], w, b, h[:m], bs, sub), y[:m]), m
        assert torch.equal(k.gemm_dx(x[:m], wt, h[:m], ats, sub), nn[:m]), m
        if K % 16 == 0:
            assert torch.equal(k.gemm_fwd_fp8(xq[:m], xs[:m].contiguous(), wq, ws, b, h[:m], bs, sub), y8[:m]), m


@pytest.mark.parametrize("K", [48, 384, 464, 1008])
def test_wide_tiles_short_contractions_and_stacked_forms(pkg, dev, K):
    """N = 1536, where 128x256 tiles are chosen (2700 rows on), contractions on both sides of the rule for
    short ones (128x128 of 8 and of 4 waves below 448), e4m3 contractions of no, some and odd whole
    k-tiles, and the stacked forward and dX: rows do not depend on the tile size there either."""
    k = pkg.kernels
    g = torch.Generator().manual_seed(K)
    M, N, G, lengths, ids = 11008, 1536, 3, (500, 700, 3000, 6808), (0, 1, -1, 0)
    rand = lambda *s, std=1.0: (torch.randn(*s, generator=g) * std).to(torch.bfloat16).to(dev)  # noqa: E731
    x, w, b, h = rand(M, K), rand(N, K, std=K ** -0.5), rand(N), rand(M, R, std=0.3)
    bs = [rand(N, R, std=0.05) for _ in range(2)]
    routing = pkg.SegmentRouting.from_lengths(lengths, ids)
    y = k.gemm_fwd(x, w, b, h, bs, routing)
    rows = torch.arange(0, M, 97, device=dev)
    ref = x[rows].double() @ w.double().t() + b.double()
    adapter = torch.tensor(routing.row_adapter(), device=dev)[rows]
    for a in range(2):
        ref += torch.where((adapter == a)[:, None], h[rows].double() @ bs[a].double().t(), 0)
    assert ((y[rows].double() - ref).norm() / ref.norm()).item() <= 2e-3
    xq, xs = k.quantize_rows_fp8(x)
    wq, ws = k.quantize_rows_fp8(w)
    y8 = k.gemm_fwd_fp8(xq, xs, wq, ws, b, h, bs, routing)
    ref8 = xq[rows].double() @ wq.double().t()
    for a in range(2):
        ref8 += torch.where((adapter == a)[:, None], h[rows].double() @ bs[a].double().t(), 0)
    ref8 = ref8 * xs[rows].double()[:, None] * ws.double() + b.double()
    assert ((y8[rows].double() - ref8).norm() / ref8.norm()).item() <= 2e-3
    h3 = rand(M, G * R, std=0.3)  # three linears of 512 columns as one product; dX of three of K = 256
    ys = k.gemm_fwd_stacked(x, w, b, h3, bs, routing, N // G, R)
    wt3, at3 = rand(N, G * 256, std=0.03), [rand(N, G * R, std=0.05) for _ in range(2)]
    dys = [rand(M, 256) for _ in range(G)]
    dx = k.gemm_dx_stacked(dys, wt3, h3, at3, routing)
    for m in (1, 65, 640, 1200, 1700, 2500, 2700, 4600, 5300, 6500):
        sub = _sub(pkg, lengths, ids, m)
        assert torch.equal(k.gemm_fwd(x[:m], w, b, h[:m], bs, sub), y[:m]), m
        assert torch.equal(k.gemm_fwd_fp8(xq[:m], xs[:m].contiguous(), wq, ws, b, h[:m], bs, sub), y8[:m]), m
        for got, want in zip(k.gemm_fwd_stacked(x[:m], w, b, h3[:m], bs, sub, N // G, R), ys):
            assert torch.equal(got, want[:m]), m
        assert torch.equal(k.gemm_dx_stacked([d[:m] for d in dys], wt3, h3[:m], at3, sub), dx[:m]), m
