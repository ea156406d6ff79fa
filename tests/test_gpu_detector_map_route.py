"""The linear index maps of gx_detector_accumulate_ws against the plain kernels of
gx_detector_accumulate, bit for bit, at sizes that the size rule sends to the maps: every case
asserts from the work size that the maps ran.  Both map kernels (the cooperative one from 160
orientations and up to 2^19 pixels, else one wave per 2 x 64 pixels), remainders of their groups
of four orientations and chunks of sixteen, and every kind of sample that leaves the map for the
exact chain: voxel planes through pixels, coordinates beyond the fixed-point range, values that
are not finite, general rotations."""

import ctypes

import numpy as np
import pytest
import torch

from giwaxsim_amd import engine
from giwaxsim_amd._lib import GxDetector, call

pytestmark = pytest.mark.gpu

# (pixels, orientations) on the map side: cooperative, direct
COOP, DIRECT = (50, 165), (52, 43)


def _images(plan, iq, q_min, dq, h=None, v=None, orient_R=None):
    """(plain image, image by ws, whether ws took the maps)."""
    t = lambda a: torch.as_tensor(np.ascontiguousarray(a, dtype=np.float64)).to('cuda')
    n = plan.n_pix
    buf = dict(h_axis=t(plan.h if h is None else h), v_axis=t(plan.v if v is None else v), init_R=t(plan.init_R),
               orient_R=t(plan.orient_R if orient_R is None else orient_R), orient_w=t(plan.orient_w))
    out, mapped = [], None
    for ws in (False, True):
        det = torch.full((n, n), -7.0, dtype=torch.float64, device='cuda')
        d = GxDetector(n_pix=n, n_init=len(buf['init_R']), n_orient=len(plan.orient_w), iq=iq.data_ptr(),
                       iq_f64=int(iq.dtype == torch.float64), cy=iq.shape[0], cx=iq.shape[1], cz=iq.shape[2],
                       qx_min=q_min[0], qy_min=q_min[1], qz_min=q_min[2], dq=dq, det=det.data_ptr(),
                       **{k: a.data_ptr() for k, a in buf.items()})
        if ws:
            work = engine.detector_work(d)
            mapped = work is not None
            call("gx_detector_accumulate_ws", ctypes.byref(d), engine.ptr(work), engine.stream_handle())
        else:
            call("gx_detector_accumulate", ctypes.byref(d), engine.stream_handle())
        out.append(det.cpu().numpy())
    return out[0], out[1], mapped


def _grid(shape, dtype, seed=0):
    g = torch.Generator(device='cuda').manual_seed(seed)
    return torch.rand(shape, generator=g, device='cuda', dtype=dtype)


def _plan(n, psis, phis=(0.0,), thetas=(0.0,), init='tilt', max_q=1.7):
    vals, axs = ((0.15,), ('psi',)) if init == 'tilt' else ((90.0, 90.0, 90.0), ('psi', 'phi', 'psi'))
    angles = [np.asarray(a, dtype=float) for a in (psis, phis, thetas)]
    w = [np.random.default_rng(3).uniform(size=len(a)) for a in angles]
    return engine.detector_plan(n, max_q, vals, axs, angles[0], w[0] / w[0].sum(), angles[1], w[1] / w[1].sum(),
                                angles[2], w[2] / w[2].sum())


@pytest.mark.parametrize("n_pix,n_orient", [
    (2, 160), (34, 161), (50, 163), (50, 175), (64, 176), (66, 257),        # cooperative
    (2, 40), (34, 41), (50, 42), (130, 43), (66, 47), (50, 63),             # direct
    (364, 66), (724, 65), (726, 67), (1026, 33), (601, 97), (727, 65),      # around 2^17 and 2^19 pixels, odd edges
])
@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
def test_sizes(n_pix, n_orient, dtype):
    print(f"[gpu-detector-route] {n_pix} px, {n_orient} orientations, {dtype}", flush=True)
    a, b, mapped = _images(_plan(n_pix, np.linspace(0.0, 173.0, n_orient)), _grid((61, 47, 83), dtype),
                           (-1.1, -1.5, -2.0), 0.0483)
    assert mapped
    assert np.array_equal(a, b)


@pytest.mark.parametrize("n_pix,n_orient", [(34, 39), (34, 64), (34, 159), (362, 64), (51, 300), (289, 500), (291, 350),
                                            (601, 92)])
def test_refused_sizes(n_pix, n_orient):
    print(f"[gpu-detector-route] refused: {n_pix} px, {n_orient} orientations", flush=True)
    a, b, mapped = _images(_plan(n_pix, np.linspace(0.0, 173.0, n_orient)), _grid((61, 47, 83), torch.float64),
                           (-1.1, -1.5, -2.0), 0.0483)
    assert not mapped
    assert np.array_equal(a, b)


@pytest.mark.parametrize("init", ['tilt', 'stand'])
@pytest.mark.parametrize("angles", [(43, 1, 1), (165, 1, 1), (21, 8, 1), (22, 1, 2), (7, 3, 8)])
def test_planes_on_boundaries(init, angles):
    """A symmetric grid of an odd edge has a voxel boundary through q = 0.  The detector's axes
    hold 0 twice, so planes that contain an axis lie on it: for all orientations, some of them
    or single lines."""
    n_psi, n_phi, n_theta = angles
    print(f"[gpu-detector-route] boundaries: {init}, {angles}", flush=True)
    q = np.linspace(-2.0, 2.0, 101)
    plan = _plan(52, np.linspace(0.0, 180.0, n_psi), np.linspace(0.0, 90.0, n_phi), np.linspace(0.0, 3.0, n_theta), init,
                 1.96)
    axis = np.concatenate([np.linspace(-1.96, 0.0, 26), np.linspace(0.0, 1.96, 26)])
    a, b, mapped = _images(plan, _grid((101, 101, 101), torch.float64), (q[0],) * 3, float(np.diff(q)[0]), h=axis, v=axis)
    assert mapped
    assert np.array_equal(a, b)


def test_odd_image_on_boundaries():
    """An odd image on the map side: its own middle row and column lie at q = 0."""
    print("[gpu-detector-route] 401 px, 9 psi x 24 phi, stand", flush=True)
    q = np.linspace(-2.0, 2.0, 101)
    plan = _plan(401, np.linspace(0.0, 90.0, 9), np.linspace(0.0, 179.0, 24), (0.0,), 'stand', 1.96)
    assert 0.0 in plan.h and 0.0 in plan.v
    a, b, mapped = _images(plan, _grid((101, 101, 101), torch.float64), (q[0],) * 3, float(np.diff(q)[0]))
    assert mapped
    assert np.array_equal(a, b)


@pytest.mark.parametrize("size", [COOP, DIRECT])
@pytest.mark.parametrize("kind", ['lattice', 'outside', 'far', 'inf', 'nan_axis', 'nan_grid', 'big_matrix', 'nan_matrix',
                                  'offset'])
def test_exact_chain(kind, size):
    n, n_orient = size
    print(f"[gpu-detector-route] {kind}: {n} px, {n_orient} orientations", flush=True)
    rng = np.random.default_rng(1)
    plan = _plan(n, np.linspace(0.0, 180.0, n_orient), init='stand', max_q=0.56)
    iq, q0, dq, more = _grid((17, 17, 17), torch.float64), (-0.56,) * 3, 0.07, {}
    line = np.linspace(-0.5, 0.5, n)
    if kind == 'lattice':       # every pixel on voxel edges at psi 0, 90, 180
        more = dict(h=np.arange(n) * 0.07 / 3 - 0.56, v=np.arange(n) * 0.07 / 3 - 0.56)
    elif kind == 'outside':     # clipped on all sides
        more = dict(h=np.linspace(-3.0, 3.0, n), v=np.linspace(-2.0, 4.0, n))
    elif kind == 'far':         # beyond the fixed-point range
        more = dict(h=np.linspace(-3e3, 3e3, n), v=np.linspace(-2.0, 4e5, n))
    elif kind == 'inf':         # finite, but beyond every range
        line[7] = 1e300
        more = dict(h=line)
    elif kind == 'nan_axis':
        line[9], line[11] = np.nan, np.inf
        more = dict(v=line)
    elif kind == 'nan_grid':
        iq[3, 4, 5], iq[8, 8, 8] = float('nan'), float('inf')
    elif kind == 'big_matrix':  # intermediate coordinates 2^20 times the final ones
        R = plan.orient_R.copy()
        R[::3, :9] *= 2.0 ** 20
        R[::3, 9:18] *= 2.0 ** -20
        more = dict(orient_R=R)
    elif kind == 'nan_matrix':
        R = plan.orient_R.copy()
        R[5, 4], R[5, 13], R[6, 2] = 1e308, 1e-308, np.nan
        more = dict(orient_R=R)
    else:                       # no symmetry: origin and rotations at random
        q0 = tuple(rng.uniform(-0.6, -0.5, 3))
        Q = np.stack([np.linalg.qr(rng.normal(size=(3, 3)))[0].ravel() for _ in range(3 * n_orient)])
        more = dict(orient_R=Q.reshape(n_orient, 27))
    a, b, mapped = _images(plan, iq, q0, dq, **more)
    assert mapped
    assert np.array_equal(a, b, equal_nan=True)


def test_grid_beyond_two_gib():
    """Byte offsets of the maps' gathers beyond 2^31: an FP64 grid of 647^3, zero below them."""
    print("[gpu-detector-route] 647^3 FP64 grid, 300 px, 181 orientations", flush=True)
    iq = _grid((647, 647, 647), torch.float64)
    low = 642  # first index whose whole slab lies beyond
    assert low * 647 * 647 * 8 >= 2 ** 31
    iq[:low] = 0.0
    q = np.linspace(-2.0, 2.0, 647)
    a, b, mapped = _images(_plan(300, np.linspace(0.0, 180.0, 181), max_q=2.1), iq, (q[0],) * 3, float(np.diff(q)[0]))
    assert mapped
    assert np.count_nonzero(a) > 1000
    assert np.array_equal(a, b)
