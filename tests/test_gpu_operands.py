"""Adapter operands made in one launch (hi / lo parts, padding, stacking, transposes) against the
torch conversions, bit for bit: both are defined roundings. Shapes at the edges of the 64x64 tiles, more
matrices than one launch takes, outputs inside wider buffers, special values."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def bits(t):
    return t.contiguous().view(torch.int16)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("pad", [8, 3])  # 16-byte accesses, and rows that do not allow them
@pytest.mark.parametrize("shapes", [[(8, 8)], [(128, 1536), (72, 72)], [(64, 64), (65, 63), (1, 129), (0, 16)], [(5, 200)] * 70])
def test_prepared_operands_are_the_torch_conversions(pkg, dev, dtype, shapes, pad):
    k = pkg.kernels
    g = torch.Generator().manual_seed(len(shapes))
    srcs, his, los, ts = [], [], [], []
    for i, (r, c) in enumerate(shapes):
        wide = (torch.randn(r, c + pad, generator=g) * 10.0 ** (i % 7 - 3)).to(dev, dtype)
        if r:
            wide[0, 0] = [float("inf"), float("-inf"), 0.0, 1e-40, -0.0][i % 5]
        srcs.append(wide[:, :c])
        pr, pc = (r + 7) // 8 * 8, (c + 7) // 8 * 8
        hi, lo, t = (torch.full(s, -1.0, dtype=torch.bfloat16, device=dev) for s in ((pr, pc + 8), (pr, pc + 8), (pc, pr + pad)))
        his.append(hi[:, :pc])
        los.append(lo[:, :pc])
        ts.append(t[:, :pr])
    k.prepare_operands(srcs, hi=his, lo=los, t=ts)
    for s, hi, lo, t in zip(srcs, his, los, ts):
        r, c = s.shape
        want = torch.zeros(hi.shape, dtype=torch.bfloat16, device=dev)
        want_lo = torch.zeros_like(want)
        want[:r, :c] = s.to(torch.bfloat16)
        want_lo[:r, :c] = (s.float() - want[:r, :c].float()).to(torch.bfloat16)
        finite = torch.isfinite(want.float())  # inf - inf: not a number on both sides, of any payload
        assert torch.equal(bits(hi), bits(want)) and torch.equal(bits(t), bits(want.t()))
        assert torch.equal(lo[finite], want_lo[finite])
    outs = k.transpose_many([h.contiguous() for h in his])
    assert all(torch.equal(bits(o), bits(h.t())) for o, h in zip(outs, his))


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("form", ["one_row", "expanded", "far_rows"])
def test_adapters_of_any_pitch_are_taken(pkg, dev, dtype, form):
    """A rank-1 lora_a that is a transposed column (pitch 1), one of equal rows (pitch 0) and a rank-1 one
    with a pitch past 32 bits: the call is the one on contiguous copies."""
    K, N = 96, 64
    g = torch.Generator().manual_seed(3)

    def rand(*shape):
        return torch.randn(*shape, generator=g).to(dev)

    if form == "far_rows":
        a = rand(1, K).to(dtype).as_strided((1, K), (2 ** 31, 1))
    else:
        a = rand(K, 1).to(dtype).t() if form == "one_row" else rand(1, K).to(dtype).expand(4, K)
    r = a.shape[0]
    assert a.stride(0) < K or a.stride(0) >= 2 ** 31
    x, w, b = rand(40, K).bfloat16(), rand(N, K).bfloat16(), rand(N, r).to(dtype)
    routing = pkg.SegmentRouting.from_lengths([40], [0])
    got, want = (pkg.multi_lora_linear(x, w, None, [m], [b], [1.0], routing)
                 for m in (a, a.clone(memory_format=torch.contiguous_format)))
    assert torch.equal(got, want)


@pytest.mark.parametrize("path", ["bf16", "f32", "fp8", "gated", "shared"])
def test_one_row_of_a_wider_matrix_is_taken(pkg, dev, path):
    """A single row x [1, K] counts as contiguous at any pitch; the call is the one on a copy."""
    K, N, r = 64, 256, 16
    g = torch.Generator().manual_seed(5)
    dt = torch.float32 if path == "f32" else torch.bfloat16

    def rand(*shape, dtype=dt):
        return torch.randn(*shape, generator=g).to(dev, dtype)

    x, res, up = rand(1, K + 1)[:, :K], rand(1, N + 3, dtype=torch.float32)[:, :N], rand(1, N)
    assert x.stride(0) == K + 1 and x.is_contiguous()
    w, a, b, gate = rand(N, K), rand(r, K), rand(N, r), rand(1, N, dtype=torch.float32)
    routing = pkg.SegmentRouting.single(1)

    def call(x, res):
        ls = [t.clone().requires_grad_(True) for t in (a, b)]
        leaf = x.detach().requires_grad_(True)
        if path == "fp8":
            y = pkg.multi_lora_linear_fp8(leaf, *pkg.kernels.quantize_rows_fp8(w), None, ls[:1], ls[1:], [1.0], routing)
        elif path == "gated":
            y = pkg.multi_lora_linear_gated(leaf, w, None, ls[:1], ls[1:], [1.0], routing, res, gate)
        elif path == "shared":
            y = sum(pkg.shared_input_multi_lora(leaf, [w, w], [None] * 2, [ls[:1]] * 2, [ls[1:]] * 2, [1.0], routing))
        else:
            y = pkg.multi_lora_linear(leaf, w, None, ls[:1], ls[1:], [1.0], routing)
        return [y.detach(), *torch.autograd.grad(y, [leaf, *ls], up.to(y.dtype))]

    for got, want in zip(call(x, res), call(x.reshape(-1).clone().view(1, K), res.reshape(-1).clone().view(1, N))):
        assert torch.equal(got, want)
