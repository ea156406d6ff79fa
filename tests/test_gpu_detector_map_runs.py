"""gx_detector_adjoint_mapped on hand-made transpose maps against exact integer sums: run
counts around a wave's chunk of 256, voxels of one run and of many chunks, uniform and mixed
orientation weights, and a run-length array at an odd address.  Equality is exact."""

import ctypes

import numpy as np
import pytest
import torch

from giwaxsim_amd._lib import GxDetector, call
from giwaxsim_amd.engine import ptr, stream_handle

pytestmark = pytest.mark.gpu

N_PIX, N_ORIENT, NV = 40, 9, (5, 7, 6)


def _runs(n, spread, rng):
    """n voxel-sorted runs inside segments of 64 pixels; few or many voxels."""
    nv = int(np.prod(NV))
    vox = np.sort(rng.integers(0, nv if spread else 3, n)).astype(np.int32)
    p = rng.integers(0, N_PIX * N_PIX, n)
    ln = np.minimum(rng.integers(1, 6, n), 64 - p % 64)
    ln[rng.random(n) < 0.02] = 0
    ln = np.where(ln == 0, 64 - p % 64, ln)
    ln = np.minimum(ln, N_PIX * N_PIX - p)
    return vox, p, ln.astype(np.uint8), rng.integers(0, N_ORIENT, n)


@pytest.mark.parametrize("mixed", [False, True])
@pytest.mark.parametrize("n,spread", [(1, False), (3, True), (255, True), (256, False), (257, True),
                                      (1024, True), (5000, False), (5001, True)])
def test_runs_sum_exactly(n, spread, mixed):
    print(f"[gpu-detector-map-runs] {n} runs, {'all' if spread else '3'} voxels, mixed weights {mixed}", flush=True)
    rng = np.random.default_rng(n)
    vox, p, ln, o = _runs(n, spread, rng)
    npx = N_PIX * N_PIX
    pbits = int(np.ceil(np.log2(npx)))
    dev = torch.device('cuda')
    w = np.full(N_ORIENT, 0.3)
    if mixed:
        w[1::2] = rng.uniform(0.1, 0.5, len(w[1::2]))
    g = rng.normal(size=npx)
    t = lambda a: torch.as_tensor(a).to(dev)
    w_d, g_d = t(w), t(g)
    vox_d = t(vox)
    ids_d = t(((o.astype(np.int64) << pbits) | p).astype(np.int32))
    len_d = torch.zeros(n + 1, dtype=torch.uint8, device=dev)[1:]  # odd address
    len_d.copy_(t(ln))
    work = torch.empty(3 * npx + (npx + 255) // 256, dtype=torch.float64, device=dev)
    det = torch.zeros(npx, dtype=torch.float64, device=dev)
    fx = torch.empty(int(np.prod(NV)), dtype=torch.int64, device=dev)
    sc = torch.empty(1, dtype=torch.float64, device=dev)
    d = GxDetector(n_pix=N_PIX, n_orient=N_ORIENT, orient_w=ptr(w_d).value, cy=NV[0], cx=NV[1], cz=NV[2], dq=1.0,
                   det=ptr(det).value)
    call("gx_detector_adjoint_mapped", ctypes.byref(d), ptr(g_d), 0, ptr(work), ptr(vox_d), ptr(ids_d), ptr(len_d), n,
         ptr(fx), ptr(sc), stream_handle())
    torch.cuda.synchronize()
    scale = float(sc.item())
    want = np.zeros(int(np.prod(NV)), dtype=np.int64)
    for k in range(n):
        q = slice(int(p[k]), int(p[k]) + int(ln[k]))
        want[vox[k]] += np.rint((g[q] * w[o[k]]) * scale).astype(np.int64).sum()
    assert np.array_equal(fx.cpu().numpy(), want)
