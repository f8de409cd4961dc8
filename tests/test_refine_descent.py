"""Barzilai-Borwein descent of the shift refinements, on the CPU."""
import torch

from artiatomi_amd.autograd import _bb_descent

F64 = torch.float64


def test_step_lengths_are_barzilai_borweins():
    """Quadratics with curvatures 1 .. 20 from a first step 1e-4 of the way: the step length has to grow several
    thousandfold at once.  Rows are compared until their gradient changes by less than float rounding of the
    largest one; the iterates agree within double rounding times the steps' curvature ratios."""
    gen = torch.Generator().manual_seed(3)
    h = torch.exp(3.0 * torch.rand((64, 2), generator=gen, dtype=F64))
    best = 8.0 * torch.rand((64, 2), generator=gen, dtype=F64) - 4.0
    first, most, s = 1e-3, 2.0, torch.zeros_like(best)
    seen = []
    _bb_descent(lambda x: h * (x - best), s, 8, first, most, callback=lambda k, x: seen.append(x.clone()))
    g = h * (s - best)
    alpha = first / g.norm(dim=1, keepdim=True)
    largest = g.norm(dim=1)
    live, compared = torch.ones(64, dtype=torch.bool), 0
    for k in range(1, 8):
        d = alpha * g
        dn = d.norm(dim=1, keepdim=True)
        new = s - torch.where(dn > most, d * (most / dn), d)
        assert torch.allclose(seen[k][live], new[live], rtol=1e-9, atol=1e-9)
        compared += int(live.sum())
        dg = h * (new - best) - g
        alpha = ((new - s) ** 2).sum(1, keepdim=True) / ((new - s) * dg).sum(1, keepdim=True)
        s, g = new, g + dg
        largest = torch.maximum(largest, g.norm(dim=1))
        live &= dg.norm(dim=1) > 1.01e-7 * largest
    assert compared > 300


def test_rows_stay_at_their_optimum():
    """Images rounded to float, as a projector's: near the optimum the residual is a few rounding errors or exactly
    0, its gradient flattens, and a step length taken from it throws a row out of the optimum.  An image moves by
    half a unit of its last place, 1.2e-7, within 1e-6 of a shift: gate 1e-4."""
    for seed in range(10):
        gen = torch.Generator().manual_seed(seed)
        a = 0.12 * torch.randn((64, 60, 2), generator=gen, dtype=F64)
        phase = 6.3 * torch.rand((64, 60), generator=gen, dtype=F64)
        best = 6.0 * torch.rand((64, 2), generator=gen, dtype=F64) - 3.0

        def arg(x):
            return (a * x[:, None]).sum(-1) + phase

        target = (2.0 + torch.sin(arg(best))).float()

        def grad(x):
            r = ((2.0 + torch.sin(arg(x))).float() - target).double()
            return 2.0 * ((r * torch.cos(arg(x)))[..., None] * a).sum(1)

        s = _bb_descent(grad, torch.zeros_like(best), 50, 0.1, 2.0)
        assert float((s - best).abs().max()) <= 1e-4
