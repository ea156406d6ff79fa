"""The row-major row pass at N = 2048, whose block takes one row of four neighbouring frames:
frame counts on both sides of multiples of four, both tile orders.  FP32 against the passes of
the column-major layout (row_variant bit 3), which take rows frame by frame: deposits, transforms
and bins are the same arithmetic, the sums are equal bit for bit.  FP64 (whose column-major rows
do not fit LDS at this size) against the oracle, to the deposit's int32 quantum."""

import numpy as np
import pytest
import torch

import oracle as O
from giwaxsim_amd import engine

pytestmark = pytest.mark.gpu

R, MAX_Q, N = 0.2, 2.0, 2048
QV = 2 * np.pi / (R * N) * (1 + 1e-9)


def _run(n_frames, precision, fill, smooth, variants):
    rng = np.random.default_rng(n_frames)
    coords = rng.uniform(0.0, 1.0, (4000, 3)) * (40.0, 30.0, 20.0)
    ids = rng.integers(0, 2, 4000).astype(np.int32)
    f = np.array([6.0 + 0.01j, 16.2 + 0.3j])
    out = {}
    for v in variants:
        res = engine.run_voxelgrid(coords, None, R, QV, MAX_Q, 12700.0, fill_bkg=fill, smooth=smooth, f_table=f,
                                   elem_ids=ids, frames=(7, 7 + n_frames), precision=precision, variant=v)
        assert res['plan'].N == N
        out[v] = (res['bins'].sum.clone(), res['bins'].cnt.clone(), res['iq64'].clone())
    return coords, f[ids], out


@pytest.mark.parametrize("n_frames", [1, 3, 4, 5, 10])
@pytest.mark.parametrize("fill,smooth", [(True, 3), (False, 0)])
def test_frame_groups_match_the_column_major_passes(n_frames, fill, smooth):
    print(f"[gpu-row-frames] N=2048 {n_frames} frames fp32 fill={fill} smooth={smooth}", flush=True)
    _, _, out = _run(n_frames, 'fp32', fill, smooth, (8, 0, 4))
    for v in (0, 4):
        assert torch.equal(out[v][1], out[8][1])
        assert torch.equal(out[v][0], out[8][0])


@pytest.mark.parametrize("n_frames", [1, 5])
def test_frame_groups_match_the_oracle(n_frames):
    print(f"[gpu-row-frames] N=2048 {n_frames} frames fp64 against the oracle", flush=True)
    coords, f_atoms, out = _run(n_frames, 'fp64', False, 0, (0, 4))
    g = engine.qgrid(QV, MAX_Q)
    ref = O.voxelgridmaker(coords, f_atoms, R, QV, MAX_Q, fill_bkg=False, smooth=0, phis=g.phis[7:7 + n_frames])
    s = slice(g.c_lo, g.c_lo + g.c_n)
    iq = ref['iq'] if ref['iq'].shape[0] == g.c_n else ref['iq'][s, s, s]
    m = iq > 1e-6 * iq.max()
    for v in (0, 4):
        got = out[v][2].cpu().numpy()
        assert np.array_equal(out[v][1].view(g.c_n, g.c_n, g.c_n).cpu().numpy(), ref['count'][s, s, s])
        assert float(np.max(np.abs(got[m] - iq[m]) / iq[m])) <= 1e-5
