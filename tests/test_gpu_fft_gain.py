"""FP32 transforms against FP64 ones in dL/df of the differentiable path, where the errors that all
frames share add up: dL/df is the difference of the atoms' part (four FP32 transforms) and the
background's (two), about 60 times as large, so a mean gain of 1 - g per transform shows as 60 g.
The FP32 constants' mean gain is within 6e-9 of 1 for the plans these edges take in both passes
(bar 4e-7); with the nearest FP32 value of cos(pi / 8) it is 3.2e-8 and dL/df is 2e-6 off."""

import numpy as np
import pytest
import torch

from giwaxsim_amd.adjoint import DifferentiableSlab

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,r,size,n", [(1024, 0.2, (60.0, 55.0, 65.0), 20000), (2048, 0.15, (50.0, 40.0, 60.0), 15000)])
def test_f_gradient(N, r, size, n):
    print(f"[gpu-fft-gain] N={N}, {n} atoms", flush=True)
    rng = np.random.default_rng(1)
    p = rng.uniform(0.0, 1.0, (n, 3)) * size
    el = np.array(['C', 'H', 'N', 'O', 'S'])[rng.choice(5, n, p=[.5, .4, .03, .03, .04])]
    det = dict(num_pixels=96, max_q=2.0, psis=np.linspace(0, 90, 19), phis=[0.0], thetas=[0.0],
               angle_init_vals=(0.15,), angle_init_axs=('psi',), mirror=True)
    h = torch.linspace(-2.0, 2.0, 96, device='cuda', dtype=torch.float64)
    q = (h[:, None] ** 2 + h[None, :] ** 2).sqrt()
    keep, scale, got = (q > 0.3).double(), None, {}
    for precision in ('fp64', 'fp32'):
        m = DifferentiableSlab(el, p, r, 2 * np.pi / (r * N) * (1 + 1e-9), 2.0, det, energy=12700.0, fill_bkg=True,
                               smooth=8, precision=precision)
        assert m.plan.N == N
        c = torch.tensor(p, device='cuda', requires_grad=True)
        f = m.f_re0.clone().requires_grad_()
        image = m(c, f, m.f_im0.clone()).double() * keep
        if scale is None:
            scale = 1.0 / float(image.max())
            target = image.detach() * (1.0 + 0.5 * torch.cos(6.0 * q))
        got[precision] = torch.autograd.grad(((scale * (image - target)) ** 2).sum(), f)[0].double()
        del m
    rel = float((got['fp32'] - got['fp64']).norm() / got['fp64'].norm())
    print(f"dL/df FP32 against FP64: {rel:.2e}", flush=True)
    assert rel <= 4e-7
