"""The one-pass backward of the modulated LayerNorm (dx, component and table gradients) at the edges
of its forms: one, two and four waves per row, partly filled lane chunks, token counts off the
workgroup's chunk, several samples, both stream dtypes. Reference: the closed form in float64.

Bounds: dx in bf16 is one rounding (2^-9 relative) of a float32 result; the float32 sums of at most
700 tokens keep 1e-5 (as tests/test_gpu_norm.py asks of the separate kernels); a bf16 component
gradient is one rounding more."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def rel(got, want):
    return ((got.double() - want).norm() / want.norm()).item()


@pytest.mark.parametrize("hidden_dtype,mod_dtype", [(torch.float32, torch.float32), (torch.bfloat16, torch.bfloat16)])
@pytest.mark.parametrize("B,T,W", [
    (1, 1, 8), (3, 9, 512), (2, 129, 520), (1, 700, 1528),   # one wave per row
    (2, 33, 1544), (1, 65, 2048), (4, 17, 3072),             # two
    (1, 40, 3080), (2, 31, 4096), (1, 70, 5120)])            # four
def test_fused_backward_matches_closed_form(pkg, dev, B, T, W, hidden_dtype, mod_dtype):
    gen = torch.Generator().manual_seed(B * T + W)
    x = (1 + 2 * torch.randn(B, T, W, generator=gen)).to(dev, hidden_dtype).requires_grad_(True)
    table = (0.1 * torch.randn(1, 6, W, generator=gen)).to(dev, mod_dtype).requires_grad_(True)
    comp = (0.3 * torch.randn(B, 6, W, generator=gen)).to(dev, mod_dtype).requires_grad_(True)
    up = torch.randn(B, T, W, generator=gen).to(dev, torch.bfloat16)
    y = pkg.modulated_layer_norm(x, table, comp, 4, 2, 1e-6)
    dx, dt, dc = torch.autograd.grad(y, [x, table, comp], up)
    xd, g = x.detach().double(), up.double()
    n = xd - xd.mean(dim=2, keepdim=True)
    rstd = (n.square().mean(dim=2, keepdim=True) + 1e-6).rsqrt()
    n = n * rstd
    s = 1 + (table.detach()[0, 4] + comp.detach()[:, 4]).double().unsqueeze(1)
    gn = g * s
    dx_ref = (gn - gn.mean(dim=2, keepdim=True) - n * (gn * n).mean(dim=2, keepdim=True)) * rstd
    dc_ref = torch.zeros(B, 6, W, dtype=torch.float64, device=dev)
    dc_ref[:, 4], dc_ref[:, 2] = (g * n).sum(1), g.sum(1)
    half = 2.0 ** -9
    # the bf16 modulation is rounded once more where table + component is added (RN of the sum)
    assert rel(dx, dx_ref) <= (1e-5 if hidden_dtype == torch.float32 else 2 * half)
    assert rel(dc, dc_ref) <= (1e-5 if mod_dtype == torch.float32 else half)
    assert rel(dt, dc_ref.sum(0, keepdim=True)) <= (1e-5 if mod_dtype == torch.float32 else half)
    assert not dc[:, [0, 1, 3, 5]].any()
    # dx does not depend on which of the other gradients are asked for (the separate hidden backward)
    (alone,) = torch.autograd.grad(pkg.modulated_layer_norm(x, table.detach(), comp.detach(), 4, 2, 1e-6), [x], up)
    assert rel(dx, alone.double()) <= (1e-6 if hidden_dtype == torch.float32 else half)
    again = torch.autograd.grad(pkg.modulated_layer_norm(x, table, comp, 4, 2, 1e-6), [x, table, comp], up)
    assert all(torch.equal(a, b) for a, b in zip((dx, dt, dc), again))


@pytest.mark.parametrize("B,T,W", [
    (5, 9, 520),       # two groups of samples, the last of one
    (64, 3, 1536), (64, 129, 72), (512, 1, 264), (512, 40, 16),
    (1024, 2, 8), (1025, 2, 8), (1290, 1, 24)])  # groups of four; of five; a last group of less
@pytest.mark.parametrize("mod_dtype", [torch.float32, torch.bfloat16])
def test_component_and_table_gradients_of_many_samples(pkg, dev, B, T, W, mod_dtype):
    """Bounds: as above for the component gradient (float32 sums over the tokens, one rounding); the
    table's float32 sum of at most 1290 of them is within sqrt(1290)·2^-24 = 2e-6 for random signs."""
    gen = torch.Generator().manual_seed(B + T + W)
    x = (1 + 2 * torch.randn(B, T, W, generator=gen)).to(dev).requires_grad_(True)
    table = (0.1 * torch.randn(1, 6, W, generator=gen)).to(dev, mod_dtype).requires_grad_(True)
    comp = (0.3 * torch.randn(B, 6, W, generator=gen)).to(dev, mod_dtype).requires_grad_(True)
    up = torch.randn(B, T, W, generator=gen).to(dev, torch.bfloat16)
    y = pkg.modulated_layer_norm(x, table, comp, 1, 5, 1e-6)
    dt, dc = torch.autograd.grad(y, [table, comp], up, retain_graph=True)
    xd, g = x.detach().double(), up.double()
    n = xd - xd.mean(dim=2, keepdim=True)
    n = n * (n.square().mean(dim=2, keepdim=True) + 1e-6).rsqrt()
    ref = torch.zeros(B, 6, W, dtype=torch.float64, device=dev)
    ref[:, 1], ref[:, 5] = (g * n).sum(1), g.sum(1)
    tol = 1e-5 if mod_dtype == torch.float32 else 2.0 ** -9
    assert rel(dc, ref) <= tol and rel(dt, ref.sum(0, keepdim=True)) <= tol
    assert not dc[:, [0, 2, 3, 4]].any() and not dt[:, [0, 2, 3, 4]].any()
    for k, one in ((0, [table]), (1, [comp])):  # either gradient alone is the same
        y1 = pkg.modulated_layer_norm(x, table if k == 0 else table.detach(), comp if k == 1 else comp.detach(), 1, 5, 1e-6)
        assert torch.equal(torch.autograd.grad(y1, one, up)[0], (dt, dc)[k])


def _gpu_us(fn, n=5):
    """GPU time of fn: the fastest of n calls, each queued behind a spinning kernel."""
    times = []
    for _ in range(n + 1):
        e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        torch.cuda._sleep(4_000_000)
        e0.record()
        fn()
        e1.record()
        e1.synchronize()
        times.append(e0.elapsed_time(e1) * 1e3)
    return min(times[1:])


@pytest.mark.parametrize("B,T,W", [(512, 8, 1536), (4096, 1, 1536), (2048, 64, 256)])
def test_many_short_samples_take_no_longer_than_the_separate_kernels(pkg, dev, B, T, W):
    """One pass over the rows must not lose to the hidden backward, the reduced component gradient and the
    sum over the samples as separate kernels where the samples are many and short (walking the samples one
    after another took 3 to 10 times as long there). Margin: 1.5, for the boxes' clocks."""
    x, up = torch.randn(B, T, W, device=dev), torch.randn(B, T, W, device=dev).bfloat16()
    table, comp = torch.randn(1, 6, W, device=dev), torch.randn(B, 6, W, device=dev)
    dx, d_comp, d_table = torch.empty_like(x), torch.empty_like(comp), torch.empty_like(table)
    mean, rstd = (torch.empty(B, T, device=dev) for _ in range(2))

    def fused():
        pkg.kernels.modulated_norm_backward_fused(x, up, comp[:, 1], table[0, 1], dx, d_comp, d_table, scale_index=1,
                                                  shift_index=0, eps=1e-6)

    def separate():
        pkg.kernels.modulated_norm_backward(x, up, comp[:, 1].unsqueeze(1).expand(B, T, W), dx, mean, rstd, eps=1e-6,
                                            scale_row=table[0, 1])
        pkg.kernels.modulated_norm_component_grad(x, up, mean, rstd, d_comp, 1, 0)
        d_comp.sum(dim=0, keepdim=True)

    assert _gpu_us(fused) <= 1.5 * _gpu_us(separate)
