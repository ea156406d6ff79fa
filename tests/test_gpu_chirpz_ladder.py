"""Every form of the wave-level chirp-z passes (length 1024) against the general, block-wide passes
of length 2048 on the same slab: the first butterflies for 2, 4, .. 16 groups of 64 inputs, bands of
up to 4, 8, 12 and 16 groups, one value to either side of their lines, FP32 and FP64, forward and
differentiable.  Both deposit the same integers."""

import numpy as np
import pytest
import torch

import test_gpu_chirpz_wave_adjoint as autograd

from giwaxsim_amd import adjoint, engine

pytestmark = pytest.mark.gpu


def _slab(size, n, seed):
    rng = np.random.default_rng(seed)
    p = rng.uniform(0.0, 1.0, (n, 3)) * np.asarray(size)
    p[:2] = [[0.0, 0.0, 0.0], size]
    return p, rng.integers(0, 2, n).astype(np.int32), np.array([6.0 + 0.01j, 16.2 + 0.3j])


def _length_2048(monkeypatch, module):
    """Chirp-z bands of length 2048, also where 1024 would do."""
    def tables(N, k_lo, K, f64=False, support=None):
        M = 2048
        t = np.arange(-(min(N, M - K + 1) - 1), K, dtype=np.int64)
        b = np.zeros(M, dtype=np.complex128)
        b[t % M] = np.exp(1j * np.pi * (((k_lo + t) ** 2) % (2 * N)) / N)
        H = (np.fft.fft(b) / M).view(np.float64)
        return M, H.astype(np.float64 if f64 else np.float32), engine.twiddles(M, f64)
    monkeypatch.setattr(module, 'chirpz_band_tables', tables)


# the row band holds 2 sqrt(2) max_q / q_voxel frequencies, the column band 2 max_q / q_voxel
def _max_q(N, r, row_band):
    return row_band / (2 * np.sqrt(2.0)) * (2 * np.pi / (r * N))


def _form(n, step):
    return min(16, max(1, -(-(-(-n // 64)) // step)) * step)


# (size in voxels, N, row band, fill, smooth, precision): (row inputs, row band, rows, column band)
FORWARD = [
    ((60, 50, 100), 600, 250, True, 3, 'fp32', (2, 4, 2, 4)),
    ((60, 50, 136), 600, 262, True, 3, 'fp32', (2, 8, 4, 4)),
    ((120, 70, 250), 600, 385, True, 0, 'fp64', (4, 8, 4, 8)),
    ((200, 150, 264), 600, 400, True, 4, 'fp32', (4, 8, 6, 8)),
    ((250, 200, 380), 600, 505, False, 0, 'fp64', (6, 8, 6, 8)),
    ((300, 200, 390), 600, 525, True, 2, 'fp32', (6, 12, 8, 8)),
    ((380, 250, 500), 600, 520, True, 0, 'fp32', (8, 12, 8, 8)),
    ((400, 350, 516), 600, 300, True, 3, 'fp32', (10, 8, 10, 4)),
    ((450, 420, 520), 700, 300, True, 3, 'fp64', (10, 8, 10, 4)),
    ((500, 420, 632), 700, 200, True, 0, 'fp32', (12, 4, 10, 4)),
    ((560, 500, 648), 800, 200, False, 0, 'fp64', (12, 4, 12, 4)),
    ((640, 540, 760), 900, 150, True, 2, 'fp32', (14, 4, 12, 4)),
    ((680, 560, 776), 1000, 100, True, 0, 'fp32', (14, 4, 14, 4)),
    ((700, 620, 900), 1000, 60, True, 0, 'fp32', (16, 4, 16, 4)),
    ((60, 50, 100), 600, 300, False, 3, 'fp32', (2, 8, 2, 4)),        # background on every row
    ((100, 90, 100), 1000, 775, True, 3, 'fp32', (4, 16, 2, 12)),
]


@pytest.mark.parametrize("voxels,N,band,fill,smooth,precision,form", FORWARD)
def test_forward(monkeypatch, voxels, N, band, fill, smooth, precision, form):
    r = 0.2
    max_q = _max_q(N, r, band)
    print(f"[gpu-chirpz-ladder] {voxels} N={N} band {band} fill={fill} smooth={smooth} {precision}", flush=True)
    coords, ids, f = _slab(np.array(voxels) * r, 3000, N)
    qv = 2 * np.pi / (r * N) * (1 + 1e-9)
    F = len(engine.qgrid(qv, max_q).phis)
    diag = int(F * np.degrees(np.arctan2(voxels[0], voxels[1])) / 180)  # the widest projection
    windows = [(0, 1), (diag, diag + 1), (F // 4, F // 4 + 1), (F // 2, F // 2 + 1)]
    angle = np.radians(engine.qgrid(qv, max_q).phis[[w[0] for w in windows]])
    y = np.outer(coords[:, 0], np.sin(angle)) + np.outer(coords[:, 1], np.cos(angle))
    top = int(np.max(np.ptp(y, axis=0) // r))
    got = []
    for length, prec in [(1024, precision), (2048, 'fp64')]:
        engine._WORKSPACES.clear()
        if length == 2048:
            _length_2048(monkeypatch, engine)
        res = engine.run_voxelgrid(coords, None, r, qv, max_q, 12700.0, fill_bkg=fill, smooth=smooth, f_table=f,
                                   elem_ids=ids, frames=windows, precision=prec)
        d = res['runner'].desc
        assert d.N == N and d.bs_M == d.bs_Mc == length
        if length == 1024:
            have = (_form(top + 1, 2), _form(d.bs_rk, 4), _form(d.Z, 2), _form(d.bs_ck, 4))
            assert have == form, (have, top + 1, d.bs_rk, d.Z, d.bs_ck)
        got.append((res['iq64'].clone(), res['bins'].cnt.clone()))
    engine._WORKSPACES.clear()
    assert torch.equal(got[0][1], got[1][1])
    want = got[1][0]
    m = want > want[want > 0].median()  # (with fill the largest value stands far above the rest)
    rel = (got[0][0] - want).abs()[m] / want[m]
    rms, largest = float(rel.square().mean().sqrt()), float(rel.max())
    print(f"rms {rms:.2e}, largest {largest:.2e}", flush=True)
    assert int(m.sum()) > 1000
    assert rms <= (2e-6 if precision == 'fp32' else 1e-8)  # a lost group would be an error of order 1


@pytest.mark.parametrize("voxels,N,band,fill,smooth,precision", [
    ((60, 50, 100), 600, 250, True, 3, 'fp32'),
    ((120, 70, 136), 600, 262, False, 0, 'fp64'),
    ((200, 150, 264), 600, 400, True, 4, 'fp64'),
    ((300, 200, 380), 600, 525, True, 2, 'fp32'),
    ((400, 350, 516), 600, 300, True, 0, 'fp64'),
    ((500, 420, 640), 700, 200, True, 3, 'fp32'),
    ((640, 540, 760), 900, 150, True, 2, 'fp32'),
    ((700, 620, 900), 1000, 60, True, 0, 'fp32'),
    ((60, 50, 100), 600, 300, False, 3, 'fp32'),
    ((100, 90, 100), 900, 775, True, 3, 'fp32'),
])
def test_differentiable(monkeypatch, voxels, N, band, fill, smooth, precision):
    r = 0.2
    max_q = _max_q(N, r, band)
    print(f"[gpu-chirpz-ladder] gradient {voxels} N={N} band {band} fill={fill} smooth={smooth} {precision}", flush=True)
    coords, ids, _ = _slab(np.array(voxels) * r, 2000, N)
    el = np.array(['C', 'S'])[ids]
    qv = 2 * np.pi / (r * N) * (1 + 1e-9)
    det = dict(num_pixels=64, max_q=max_q, psis=[0.0, 30.0, 75.0], phis=[0.0], thetas=[0.0], angle_init_vals=(0.15,),
               angle_init_axs=('psi',), mirror=True)
    F = len(engine.qgrid(qv, max_q).phis)
    diag = int(F * np.degrees(np.arctan2(voxels[0], voxels[1])) / 180)
    G = torch.as_tensor(np.random.default_rng(5).normal(size=(64, 64)), device='cuda')
    got = []
    for length in (1024, 2048):
        if length == 2048:
            _length_2048(monkeypatch, adjoint)
        m = adjoint.DifferentiableSlab(el, coords, r, qv, max_q, det, frames=(diag, diag + 3),
                                       precision=precision if length == 1024 else 'fp64', fill_bkg=fill, smooth=smooth)
        assert m.plan.N == N and m.bs['M'] == m.bs['Mc'] == length
        c = torch.tensor(coords, device='cuda', requires_grad=True)
        f = m.f_re0.clone().requires_grad_()
        image = m(c, f, m.f_im0.clone())
        got.append([image.detach()] + list(torch.autograd.grad((image * G).sum(), [c, f])))
    tol = (2e-6, 1e-4) if precision == 'fp32' else (1e-10, 1e-10)
    err = [float((x - y).abs().max() / y.abs().max()) for x, y in zip(*got)]
    print("image {:.2e} coords {:.2e} f {:.2e}".format(*err), flush=True)
    assert err[0] <= tol[0] and max(err[1:]) <= tol[1]


def test_wide_band_fp64():
    """A band of nearly every frequency in FP64 at N = 1000, which no block-wide row pass has the
    LDS for: against the FP32 transforms of the same slab."""
    print("[gpu-chirpz-ladder] N=1000, whole band, FP64 against FP32", flush=True)
    r, N = 0.2, 1000
    max_q = _max_q(N, r, 950)
    coords, ids, f = _slab(np.array([40, 30, 50]) * r, 800, N)
    got = []
    for precision in ('fp64', 'fp32'):
        engine._WORKSPACES.clear()
        res = engine.run_voxelgrid(coords, None, r, 2 * np.pi / (r * N) * (1 + 1e-9), max_q, 12700.0, fill_bkg=True,
                                   f_table=f, elem_ids=ids, frames=(100, 102), precision=precision)
        assert res['runner'].desc.bs_M == 1024 and res['runner'].desc.bs_rk > 900
        got.append(res['iq64'].clone())
        del res
    engine._WORKSPACES.clear()
    m = got[0] > 1e-6 * got[0].max()
    assert float(((got[1] - got[0]).abs()[m] / got[0][m]).max()) <= 1e-5


def test_differentiable_fp64_near_2048():
    """FP64 gradients of a small crystal on a large edge, against autograd: the wave-level passes hold
    rows of 1024 nodes, where the block-wide row gradient would need 4 N.  (A filled slab of 400 atoms
    on this edge has a background 10^5 times its intensities, and the image the bins' last bit.)"""
    autograd.test_against_autograd((30.0, 20.0, 16.0), 1990, 0.2, 0.8, False, 0, 'CN', 'fp64')
