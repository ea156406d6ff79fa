"""gx_detector_accumulate_ws against gx_detector_accumulate, bit for bit: the linear index
maps (guarded, with the exact chain for samples near a voxel boundary) against the
per-sample rotations and floors, which the oracle pins.  Sizes at the edges of the pixel
tiles (16 x 4), of the gathered groups (4 orientations) and chunks (16), of the cooperative
form (64 orientations, 2^19 pixels) and of its padding; every kind of orientation that
leaves the linear map; float and double grids of uneven edges."""

import ctypes

import numpy as np
import pytest
import torch

from giwaxsim_amd import engine
from giwaxsim_amd._lib import GxDetector, call

pytestmark = pytest.mark.gpu


def _both(plan, iq, q_min, dq, h=None, v=None, init_R=None, orient_R=None):
    dev = torch.device('cuda')
    t = lambda a: torch.as_tensor(np.ascontiguousarray(a, dtype=np.float64)).to(dev)
    h, v = t(plan.h if h is None else h), t(plan.v if v is None else v)
    iR, oR = t(plan.init_R if init_R is None else init_R), t(plan.orient_R if orient_R is None else orient_R)
    ow = t(plan.orient_w)
    n, O = plan.n_pix, len(plan.orient_w)
    out = []
    for ws in (False, True):
        det = torch.full((n, n), -7.0, dtype=torch.float64, device=dev)
        d = GxDetector(n_pix=n, n_init=len(iR), n_orient=O, h_axis=h.data_ptr(), v_axis=v.data_ptr(),
                       init_R=iR.data_ptr(), orient_R=oR.data_ptr(), orient_w=ow.data_ptr(), iq=iq.data_ptr(),
                       iq_f64=int(iq.dtype == torch.float64), cy=iq.shape[0], cx=iq.shape[1], cz=iq.shape[2],
                       qx_min=q_min[0], qy_min=q_min[1], qz_min=q_min[2], dq=dq, det=det.data_ptr())
        if ws:
            work = engine.detector_work(d)
            call("gx_detector_accumulate_ws", ctypes.byref(d), engine.ptr(work), engine.stream_handle())
        else:
            call("gx_detector_accumulate", ctypes.byref(d), engine.stream_handle())
        out.append(det.cpu().numpy())
    return out


def _grid(shape, dtype, seed=0):
    g = torch.Generator(device='cuda').manual_seed(seed)
    return torch.rand(shape, generator=g, device='cuda', dtype=dtype)


def _plan(n, psis, phis, thetas, init='tilt', max_q=1.7):
    vals, axs = ((0.15,), ('psi',)) if init == 'tilt' else ((90.0, 90.0, 90.0), ('psi', 'phi', 'psi'))
    w = [np.random.default_rng(3).uniform(size=len(a)) for a in (psis, phis, thetas)]
    return engine.detector_plan(n, max_q, vals, axs, psis, w[0] / w[0].sum(), phis, w[1] / w[1].sum(), thetas,
                                w[2] / w[2].sum())


ONE = np.array([0.0])


@pytest.mark.parametrize("n_pix,n_orient,dtype", [
    (1, 1, torch.float64), (3, 4, torch.float32), (15, 5, torch.float64), (17, 63, torch.float64),
    (33, 64, torch.float32), (33, 65, torch.float64), (49, 80, torch.float64), (64, 97, torch.float64),
    (724, 64, torch.float64), (725, 64, torch.float64), (725, 9, torch.float32),
])
def test_sizes(n_pix, n_orient, dtype):
    print(f"[gpu-detector-linear] {n_pix} px, {n_orient} orientations, {dtype}", flush=True)
    a, b = _both(_plan(n_pix, np.linspace(0.0, 173.0, n_orient), ONE, ONE), _grid((61, 47, 83), dtype), (-1.1, -1.5, -2.0),
                 0.0483)
    assert np.array_equal(a, b)


@pytest.mark.parametrize("init", ['tilt', 'stand'])
@pytest.mark.parametrize("n_phi,n_theta", [(1, 1), (4, 1), (1, 2), (3, 3)])
def test_planes_on_boundaries(init, n_phi, n_theta):
    """A symmetric grid of an odd edge has a voxel boundary through q = 0: detector planes
    that contain an axis lie on it, for all orientations, some of them or single lines."""
    print(f"[gpu-detector-linear] boundaries: {init}, {n_phi} phi, {n_theta} theta", flush=True)
    q = np.linspace(-2.0, 2.0, 101)
    plan = _plan(51, np.linspace(0.0, 180.0, 37), np.linspace(0.0, 90.0, n_phi), np.linspace(0.0, 3.0, n_theta), init, 1.96)
    a, b = _both(plan, _grid((101, 101, 101), torch.float64), (q[0],) * 3, float(np.diff(q)[0]))
    assert np.array_equal(a, b)


@pytest.mark.parametrize("kind", ['lattice', 'outside', 'far', 'inf', 'nan_grid', 'big_matrix', 'nan_matrix', 'offset'])
def test_exact_chain_cases(kind):
    print(f"[gpu-detector-linear] {kind}", flush=True)
    rng = np.random.default_rng(1)
    plan = _plan(49, np.linspace(0.0, 180.0, 65), ONE, ONE, 'stand', 0.56)
    iq, q0, dq, more = _grid((17, 17, 17), torch.float64), (-0.56,) * 3, 0.07, {}
    if kind == 'lattice':      # every pixel on voxel edges at psi 0, 90, 180
        more = dict(h=np.arange(49) * 0.07 / 3 - 0.56, v=np.arange(49) * 0.07 / 3 - 0.56)
    elif kind == 'outside':    # clipped on all sides
        more = dict(h=np.linspace(-3.0, 3.0, 49), v=np.linspace(-2.0, 4.0, 49))
    elif kind == 'far':        # beyond the fixed-point range
        more = dict(h=np.linspace(-3e3, 3e3, 49), v=np.linspace(-2.0, 4e5, 49))
    elif kind == 'inf':
        h = np.linspace(-0.5, 0.5, 49)
        h[7] = 1e300
        more = dict(h=h)
    elif kind == 'nan_grid':
        iq[3, 4, 5], iq[8, 8, 8] = float('nan'), float('inf')
    elif kind == 'big_matrix':  # intermediate coordinates 2^20 times the final ones
        R = plan.orient_R.copy()
        R[::3, :9] *= 2.0 ** 20
        R[::3, 9:18] *= 2.0 ** -20
        more = dict(orient_R=R)
    elif kind == 'nan_matrix':
        R = plan.orient_R.copy()
        R[5, 4] = 1e308
        R[5, 13] = 1e-308
        more = dict(orient_R=R)
    else:                       # no symmetry: origin and rotations at random
        q0 = tuple(rng.uniform(-0.6, -0.5, 3))
        Q = np.stack([np.linalg.qr(rng.normal(size=(3, 3)))[0].ravel() for _ in range(3 * 65)]).reshape(65, 27)
        more = dict(orient_R=Q)
    a, b = _both(plan, iq, q0, dq, **more)
    assert np.array_equal(a, b, equal_nan=True)


@pytest.mark.parametrize("n_pix,n_orient", [(15, 39), (15, 40), (33, 63), (33, 64), (33, 159), (33, 160), (1, 160),
                                            (49, 163), (64, 257), (362, 64), (363, 64),
                                            (14, 40), (34, 160), (50, 163), (2, 200), (599, 41), (601, 41), (601, 64)])
@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
def test_both_sides_of_the_size_rule(n_pix, n_orient, dtype):
    """Orientation counts and image sizes at the lines where the linear maps take over from the
    plain kernels and from their cooperative form."""
    print(f"[gpu-detector-linear] rule: {n_pix} px, {n_orient} orientations, {dtype}", flush=True)
    a, b = _both(_plan(n_pix, np.linspace(0.0, 173.0, n_orient), ONE, ONE), _grid((61, 47, 83), dtype), (-1.1, -1.5, -2.0),
                 0.04)
    assert np.array_equal(a, b, equal_nan=True)
