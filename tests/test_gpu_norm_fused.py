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
