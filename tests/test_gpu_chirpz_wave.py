"""The wave-level chirp-z passes of length 1024 against the oracle: grid edges on both sides
of every rule that picks a form of them: atoms that end below 640 rows (10 of the 16 input
groups) or not, bands of up to 320 frequencies (5 of 16 output groups) or wider, row counts
on both sides of 640, with and without fill and smoothing, FP32 and FP64 transforms, and the
first edge whose band needs length 2048."""

import numpy as np
import pytest

import oracle as O
from giwaxsim_amd import engine

pytestmark = pytest.mark.gpu


def _slab(size, n, seed):
    rng = np.random.default_rng(seed)
    p = rng.uniform(0.0, 1.0, (n, 3)) * np.asarray(size)
    p[:2] = [[0.0, 0.0, 0.0], size]
    return p, rng.integers(0, 2, n).astype(np.int32), np.array([6.0 + 0.01j, 16.2 + 0.3j])


# (size, N, r, max_q, fill, smooth, precision): input groups, band groups
CASES = [
    ((20.0, 12.0, 18.0), 300, 0.25, 2.0, False, 0, 'fp64'),
    ((20.0, 12.0, 18.0), 301, 0.25, 2.0, True, 3, 'fp32'),
    ((100.0, 60.0, 20.0), 700, 0.2, 1.0, True, 0, 'fp32'),     # y_max < 640
    ((110.0, 75.0, 20.0), 700, 0.2, 1.0, True, 4, 'fp32'),     # y_max >= 640
    ((110.0, 75.0, 20.0), 700, 0.2, 1.0, False, 0, 'fp64'),
    ((30.0, 20.0, 127.8), 700, 0.2, 1.0, True, 4, 'fp32'),     # Z = 640
    ((30.0, 20.0, 130.0), 700, 0.2, 1.0, True, 4, 'fp32'),     # Z = 656
    ((30.0, 20.0, 130.0), 700, 0.2, 1.0, False, 4, 'fp32'),    # background on every row
    ((40.0, 20.0, 30.0), 600, 0.2, 3.1, True, 2, 'fp32'),      # band wider than 320
    ((40.0, 20.0, 30.0), 600, 0.2, 3.1, False, 0, 'fp64'),
    ((118.0, 90.0, 20.0), 800, 0.2, 1.2, True, 4, 'fp32'),     # support + band beyond 1024
]


@pytest.mark.parametrize("size,N,r,max_q,fill,smooth,precision", CASES)
def test_against_oracle(size, N, r, max_q, fill, smooth, precision):
    print(f"[gpu-chirpz-wave] {size} N={N} max_q={max_q} fill={fill} smooth={smooth} {precision}", flush=True)
    coords, ids, f = _slab(size, 3000, N)
    qv = 2 * np.pi / (r * N) * (1 + 1e-9)
    g = engine.qgrid(qv, max_q)
    # six windows of two frames, at the axes' and the diagonals' angles
    F = len(g.phis)
    windows = [(w, w + 2) for w in (0, F // 8, F // 4, F // 2, 3 * F // 4, F - 2)]
    res = engine.run_voxelgrid(coords, None, r, qv, max_q, 12700.0, fill_bkg=fill, smooth=smooth, f_table=f,
                               elem_ids=ids, frames=windows, precision=precision)
    assert res['plan'].N == N
    phis = np.concatenate([g.phis[a:b] for a, b in windows])
    ref = O.voxelgridmaker(coords, f[ids], r, qv, max_q, fill_bkg=fill, smooth=smooth, phis=phis)
    s = slice(g.c_lo, g.c_lo + g.c_n)
    cnt = res['bins'].cnt.view(g.c_n, g.c_n, g.c_n).cpu().numpy()
    assert np.array_equal(cnt, ref['count'][s, s, s])
    iq = res['iq64'].cpu().numpy()
    m = ref['iq'] > 1e-6 * ref['iq'].max()
    rel = float(np.max(np.abs(iq[m] - ref['iq'][m]) / ref['iq'][m]))
    print(f"max rel err {rel:.2e}", flush=True)
    assert rel <= 1e-5
