"""The shrink's mask-free loads of whole 64-wide k-tiles and its masked ones around their edges: contractions
of no, some and only whole k-tiles, more and fewer than the pipeline holds, every rank template, both
operand layouts. Appending columns of zeros to both operands adds zero products at the end of the same
sum, so h must not change by a bit; against float64, h is one bf16 rounding (2^-8 covers
it with the float32 sum's error)."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("layout", [0, 1])
@pytest.mark.parametrize("r", [16, 64, 128, 192])
@pytest.mark.parametrize("split", [False, True])
@pytest.mark.parametrize("K", [8, 56, 64, 72, 128, 192, 248, 256, 576])
def test_shrink_at_k_tile_edges(pkg, dev, K, r, layout, split):
    gen = torch.Generator().manual_seed(K + r)
    routing = pkg.SegmentRouting.from_lengths([33, 300, 32], [0, 1, 0])
    M = routing.num_rows
    x = torch.randn(M, K, generator=gen).bfloat16()
    ops = [torch.randn(r, K, generator=gen) for _ in range(2)]
    scales = [1.0, 0.5]

    def call(pad):
        wide = [torch.nn.functional.pad(o, (0, pad)) for o in ops]
        hi = [o.bfloat16() for o in wide]
        lo = [(o - h.float()).bfloat16() for o, h in zip(wide, hi)] if split else None
        lay = (lambda ts: [(t if layout == 0 else t.t()).contiguous().to(dev) for t in ts])
        return pkg.kernels.shrink(torch.nn.functional.pad(x, (0, pad)).to(dev), lay(hi), layout, scales, routing,
                                  want_frag=False, width=r, ops_lo=lay(lo) if split else None)[0]

    h = call(0)
    for pad in (8, 64):
        assert torch.equal(h.view(torch.int16), call(pad).view(torch.int16))
    used = [o if split else o.bfloat16().float() for o in ops]
    for s, (a, lo_, hi_) in enumerate(((0, 0, 33), (1, 33, 333), (0, 333, 365))):
        want = scales[a] * (x[lo_:hi_].double() @ used[a].double().t())
        got = h[lo_:hi_].cpu().double()
        assert ((got - want).norm() / want.norm()).item() <= 2.0 ** -8
