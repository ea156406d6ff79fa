"""The k = 0 column of the wave-level chirp-z path with smoothing and no fill: its background A N is
added to the transform as one value, so FP32 rows hold no multiple of it, neither those of the row
pass nor those beyond the atoms.  The central line of I(q) is then as exact, FP32 against FP64, as
the other voxels; with A N in the rows beyond the atoms its relative error is half as large again
as theirs."""

import numpy as np
import pytest

from giwaxsim_amd import engine

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("seed", [1, 2])
def test_central_line(seed):
    print(f"[gpu-chirpz-k0] N=700, 200 of 700 rows hold atoms, seed {seed}", flush=True)
    rng = np.random.default_rng(seed)
    size, N, r = (30.0, 20.0, 40.0), 700, 0.2
    p = rng.uniform(0.0, 1.0, (4000, 3)) * size
    p[:2] = [[0.0, 0.0, 0.0], size]
    ids, f = rng.integers(0, 2, 4000).astype(np.int32), np.array([6.0 + 0.01j, 16.2 + 0.3j])
    iq = {}
    for precision in ('fp64', 'fp32'):
        res = engine.run_voxelgrid(p, None, r, 2 * np.pi / (r * N) * (1 + 1e-9), 1.0, 12700.0, smooth=4, f_table=f,
                                   elem_ids=ids, precision=precision)
        assert res['plan'].N == N
        iq[precision] = res['iq64'].cpu().numpy()
    ref = iq['fp64']
    rel = np.abs(iq['fp32'] - ref) / np.where(ref > 0, ref, 1.0)
    c = ref.shape[0] // 2
    line, rest = np.delete(rel[c, c], c), ref > 0
    rest[c - 1:c + 2, c - 1:c + 2] = False
    rms = [float(np.sqrt(np.mean(x ** 2))) for x in (line, rel[rest])]
    print(f"rms relative error: central line {rms[0]:.2e}, other voxels {rms[1]:.2e}", flush=True)
    assert rms[0] <= rms[1]
