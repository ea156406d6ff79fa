"""Stable regrouping by z row (gx_slab_sort_rows with the permutation): atom counts around a
wave, a pass of 1,024 and a chunk of 4,096, grid edges with row indices of 5 to 12 bits, rows
shared by every atom and by none, atoms of no known element (the row after the last).  Exact."""

import ctypes

import numpy as np
import pytest
import torch

from giwaxsim_amd import _lib, engine
from giwaxsim_amd._lib import GxSlab, call
from giwaxsim_amd.engine import ptr

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 63, 64, 65, 1023, 1024, 1025, 4096, 4097, 9000])
@pytest.mark.parametrize("N,layers", [(16, 16), (255, 1), (256, 200), (2048, 2048)])
def test_order_is_stable(n, N, layers):
    print(f"[gpu-stable-sort] n={n} N={N} {layers} rows used", flush=True)
    rng = np.random.default_rng(n + N)
    r = 0.25
    row = rng.integers(0, layers, n)
    xyz = np.stack([rng.random(n), rng.random(n), (row + 0.5) * r])
    ids = rng.integers(0, 3, n)  # 2: beyond the element table
    ft = np.array([[6.0, 0.1], [16.0, 0.3]])
    dev = torch.device('cuda')
    t = lambda a, dt: torch.as_tensor(np.ascontiguousarray(a)).to(device=dev, dtype=dt)
    e = lambda m, dt: torch.empty(m, dtype=dt, device=dev)
    f64, i32 = torch.float64, torch.int32
    x, y, z = (t(c, f64) for c in xyz)
    el, ftab = t(ids, i32), t(ft, f64)
    sx, sy, szf, szrow, sperm, selem, sq = e(n, f64), e(n, f64), e(n, f64), e(n, i32), e(n, i32), e(n, i32), e(2 * n, i32)
    off, exp, work = e(N + 2, i32), e(N, i32), e(N * 2 + 2 * (N + 1), i32)
    stable = e(-(-n // _lib.GX_STABLE_CHUNK) * (N + 1), i32)
    p = lambda a: ptr(a).value
    d = GxSlab(n_atoms=n, n_elem=2, N=N, r=r, zmin=0.0, x=p(x), y=p(y), z=p(z), elem=p(el), f_table=p(ftab), sx=p(sx),
               sy=p(sy), sq=p(sq), szrow=p(szrow), row_off=p(off), row_exp=p(exp), work=p(work), szf=p(szf),
               sperm=p(sperm), selem=p(selem), stable_work=p(stable))
    call("gx_slab_sort_rows", ctypes.byref(d), engine.stream_handle())
    rows = np.where(ids < 2, row, N)
    want = np.lexsort((np.arange(n), rows))
    assert np.array_equal(sperm.cpu().numpy(), want)
    assert np.array_equal(szrow.cpu().numpy(), rows[want])
    assert np.array_equal(sx.cpu().numpy(), xyz[0][want])
    assert np.array_equal(sy.cpu().numpy(), xyz[1][want])
    assert np.array_equal(selem.cpu().numpy(), ids[want])
    assert np.array_equal(sq.cpu().numpy().reshape(-1, 2)[rows[want] == N], np.zeros(((rows == N).sum(), 2)))
