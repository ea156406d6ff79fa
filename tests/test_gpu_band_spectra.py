"""The background spectra of grid edges that are not powers of two (direct FP64 DFTs in groups of
eight rows, frequencies in pairs) against numpy's dense sums of the same profiles, read back from
the device: the smallest edges, every remainder by eight, even and odd.  An FP64 sum of N terms
in any order is within (N + 16) eps sum |terms| of the exact one: the bar is four times that."""

import numpy as np
import pytest
import torch

from giwaxsim_amd import _lib
from giwaxsim_amd.adjoint import DifferentiableSlab

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N", [16, 17, 18, 27, 36, 45, 54, 63, 130])
@pytest.mark.parametrize("smooth", [0, 2])
def test_spectra_against_dense_sums(N, smooth):
    print(f"[gpu-band-spectra] N={N} fill, smooth {smooth}", flush=True)
    r, max_q = 0.8, 2.4
    rng = np.random.default_rng(N)
    coords = rng.uniform(0.0, 1.0, (200, 3)) * (0.5 * r * N, 0.4 * r * N, 0.4 * r * N)
    el = np.array(['C', 'S'])[rng.integers(0, 2, 200)]
    qv = 2 * np.pi / (r * N) * (1 + 1e-9)
    det = dict(num_pixels=16, max_q=max_q, psis=[0.0, 40.0], phis=[0.0], thetas=[0.0],
               angle_init_vals=(0.15,), angle_init_axs=('psi',), mirror=True)
    m = DifferentiableSlab(el, coords, r, qv, max_q, det, frames=(0, 3), precision='fp64', fill_bkg=True,
                           smooth=smooth)
    assert m.plan.N == N and m.bs is not None and m.batch >= 3
    c = torch.tensor(coords, dtype=torch.float64, device='cuda', requires_grad=True)
    m(c, m.f_re0.clone(), m.f_im0.clone()).sum().backward()
    fr, adj = m._prepared
    # the profiles and spectra of the batch as the backward left them
    W = int(fr.W)
    f8 = lambda t: t.cpu().numpy()
    nm = f8(m.col_nm).reshape(-1, N).astype(float)
    sy = f8(m.col_sy).reshape(-1, N) if smooth else np.ones((m.batch, N))
    sz = f8(m.col_sz).reshape(-1, N) if smooth else np.ones((m.batch, N))
    bounds = f8(m.idx_bounds).reshape(-1, 4)
    spec = f8(m.col_spec).view(np.complex128).reshape(-1, W)
    both = f8(m.avg_spec).view(np.complex128).reshape(-1, N + W)
    fp = f8(m.fparams).reshape(-1, _lib.GX_FP_STRIDE)
    y = np.arange(N)
    avg, mv = complex(fr.avg_re, fr.avg_im), float(fr.max_voxels)
    for fb in range(3):
        ylo, yhi, zlo, zhi = bounds[fb]
        bkg = np.where((y > ylo) & (y < yhi), nm[fb], mv) * avg * sy[fb]
        if smooth:
            bkg = bkg - mv * avg * sy[fb]
        jlo, jhi = int(fp[fb, _lib.FP_JLO]), int(fp[fb, _lib.FP_JHI])
        kc = np.arange(jlo, jhi + 1) - N // 2
        kz = np.arange(m.bs['clo'], m.bs['clo'] + m.bs['ck'])
        pz = np.where((y >= zlo) & (y < zhi), sz[fb], 0.0)
        py = np.where((y > ylo) & (y < yhi), nm[fb] - mv, 0.0) * sy[fb]
        for name, u, k, got in (('background', bkg, kc, spec[fb, :len(kc)]), ('z', pz, kz, both[fb, kz % N]),
                                ('y', py, kc, both[fb, N:N + len(kc)])):
            phase = (np.outer(k, y) % N) * (-2j * np.pi / N)
            want = (np.exp(phase) * u).sum(1)
            bar = 4 * (N + 16) * np.finfo(float).eps * np.abs(u).sum()
            assert np.max(np.abs(got - want)) <= bar, (name, fb, np.max(np.abs(got - want)), bar)
