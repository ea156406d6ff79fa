"""The wave-level chirp-z passes of the differentiable path (bands of length 1024) against the
FP64 autograd reference, on both sides of every rule that picks a form of them: deposits that
end below 640 rows (10 of the 16 input groups) or not, bands of up to 320 frequencies (5 of 16
groups) or wider, row counts on both sides of 640, grid edges below and above 1024, with and
without fill and smoothing, up to and beyond six elements.  Bars of test_gpu_adjoint."""

import numpy as np
import pytest
import torch

from giwaxsim_amd.adjoint import DifferentiableSlab
from giwaxsim_amd.engine import element_table, qgrid
from oracle.cic_model import CicModel

pytestmark = pytest.mark.gpu

TOL = {'fp64': (1e-10, 1e-10), 'fp32': (2e-6, 1e-4)}

# (size, N, r, max_q, fill, smooth, elements, precision)
CASES = [
    ((20.0, 12.0, 18.0), 300, 0.25, 2.0, False, 0, 'CN', 'fp64'),
    ((110.0, 75.0, 12.0), 700, 0.2, 1.0, True, 4, 'CN', 'fp64'),     # y_max >= 640 at the diagonal
    ((110.0, 75.0, 12.0), 700, 0.2, 1.0, True, 0, 'CN', 'fp32'),
    ((20.0, 15.0, 127.4), 700, 0.2, 1.0, True, 4, 'CN', 'fp32'),     # Z = 640
    ((20.0, 15.0, 130.0), 700, 0.2, 1.0, True, 4, 'CN', 'fp64'),     # Z = 656
    ((30.0, 20.0, 16.0), 600, 0.2, 3.1, True, 2, 'CNOSFHB', 'fp64'),  # bands wider than 320
    ((30.0, 20.0, 16.0), 600, 0.2, 3.1, False, 0, 'CN', 'fp32'),
    ((30.0, 20.0, 16.0), 1100, 0.2, 1.0, True, 3, 'CNOSFHB', 'fp32'),
]


@pytest.mark.parametrize("size,N,r,max_q,fill,smooth,elements,precision", CASES)
def test_against_autograd(size, N, r, max_q, fill, smooth, elements, precision):
    print(f"[gpu-chirpz-wave-adjoint] {size} N={N} max_q={max_q} fill={fill} smooth={smooth} {elements} {precision}",
          flush=True)
    rng = np.random.default_rng(N)
    coords = rng.uniform(0.0, 1.0, (400, 3)) * np.asarray(size)
    coords[:2] = [[0.0, 0.0, 0.0], size]
    el = np.array(list(elements))[np.arange(400) % len(elements)]
    qv = 2 * np.pi / (r * N) * (1 + 1e-9)
    det = dict(num_pixels=32, max_q=max_q, psis=[0.0, 30.0, 75.0], phis=[0.0], thetas=[0.0],
               angle_init_vals=(0.15,), angle_init_axs=('psi',), mirror=True)
    F = len(qgrid(qv, max_q).phis)
    frames = (F // 5, F // 5 + 3)  # near the diagonal of the wide slab
    uniq = sorted(set(el))
    ids = np.array([uniq.index(e) for e in el])
    _, ftab, _, _ = element_table(el, 12700.0)
    ref = CicModel(coords, ids, r, qv, max_q, det, frames=frames, fill_bkg=fill, smooth=smooth)
    ct = torch.tensor(coords, dtype=torch.float64, requires_grad=True)
    frt = torch.tensor(ftab.real.copy(), requires_grad=True)
    fit = torch.tensor(ftab.imag.copy(), requires_grad=True)
    G = rng.normal(size=(32, 32))
    want = ref(ct, frt, fit)
    (want * torch.as_tensor(G)).sum().backward()
    model = DifferentiableSlab(el, coords, r, qv, max_q, det, frames=frames, precision=precision,
                               fill_bkg=fill, smooth=smooth)
    assert model.plan.N == N and model.bs['M'] == 1024
    dev = torch.device('cuda')
    c = torch.tensor(coords, dtype=torch.float64, device=dev, requires_grad=True)
    fr = model.f_re0.clone().requires_grad_(True)
    fi = model.f_im0.clone().requires_grad_(True)
    img = model(c, fr, fi)
    (img * torch.as_tensor(G, device=dev)).sum().backward()
    err = [float(np.max(np.abs(a.detach().cpu().numpy() - b.detach().numpy())) / np.max(np.abs(b.detach().numpy())))
           for a, b in ((img, want), (c.grad, ct.grad), (fr.grad, frt.grad), (fi.grad, fit.grad))]
    print("  image {:.2e}  d/dcoords {:.2e}  d/df_re {:.2e}  d/df_im {:.2e}".format(*err), flush=True)
    tol_img, tol_grad = TOL[precision]
    assert err[0] <= tol_img and max(err[1:]) <= tol_grad
