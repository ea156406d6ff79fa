"""The rounded constants of the FP32 transforms, on the CPU: the matrix that each radix plan
computes with its FP32 constants and twiddles but exact arithmetic, against the exact DFT.  Their
rounding acts on every frame and row alike, so it does not average out of I(q) as the rounding of
the data does.  The radix-16 constant cos(pi / 8) is the FP32 value above it rather than the nearest:
over every plan with a radix of 16, the mean gain, the rms error and the largest error of an output's
gain are no larger than with the nearest value."""

import os
import re

import numpy as np
import pytest

HEADER = os.path.join(os.path.dirname(__file__), "..", "giwaxsim_amd", "csrc", "gx_device.h")
f32 = np.float32

# the in-wave plans by length, the chirp-z plans (wave: 16.4.16, block: 8.4.8.8, 16.16.16)
PLANS = [(16, 16, 4), (16, 8, 8), (8, 16, 8), (8, 8, 16), (16, 4, 16), (16, 16, 8), (16, 8, 16), (8, 16, 16),
         (16, 16, 16)]


def _constants():
    text = open(HEADER).read()
    body = text[text.index("struct DftConst"):]
    c1 = re.search(r"c1 = sizeof\(T\) == 4 \? \(T\)([0-9.]+) : \(T\)([0-9.]+)", body)
    c2 = re.search(r"c2 = \(T\)([0-9.]+)", body)
    t = re.search(r"\bt = \(T\)([0-9.]+)", body)
    assert float(c1.group(2)) == np.cos(np.pi / 8) and float(t.group(1)) == np.tan(np.pi / 8)
    assert float(c2.group(1)) == np.sqrt(0.5)
    return [float(f32(x)) for x in (c1.group(1), c2.group(1), t.group(1))]


def _small(R, c):
    """The DFT of R values with constants (c1, c2, t) as the kernels form it."""
    if R == 4:
        return np.exp(-0.5j * np.pi * np.outer(np.arange(4), np.arange(4))).round()
    c1, c2, t = c
    half = _small(R // 2, c)
    w8 = [1, c2 * (1 - 1j), -1j, -c2 * (1 + 1j)]
    w16 = [1, c1 * (1 - 1j * t), w8[1], c1 * (t - 1j), -1j, -c1 * (t + 1j), w8[3], -c1 * (1 + 1j * t)]
    o = np.array(w8 if R == 8 else w16)[:, None] * half
    out = np.empty((R, R), dtype=complex)
    out[:, 0::2] = np.concatenate([half, half])
    out[:, 1::2] = np.concatenate([o, -o])
    return out


def _gain_error(plan, c):
    """(k, n): relative error of the transform's matrix elements."""
    N = int(np.prod(plan))
    k = np.arange(N)
    tw = np.exp(-2j * np.pi * k / N)
    tw = tw.real.astype(f32).astype(float) + 1j * tw.imag.astype(f32).astype(float)
    n = np.arange(N) if N <= 1024 else np.random.default_rng(1).choice(N, 256, replace=False)
    x = np.zeros((N, len(n)), dtype=complex)
    x[n, np.arange(len(n))] = 1.0
    done = 1
    for R in plan:
        j = np.arange(N // R)
        p = j % done
        v = np.stack([x[j + r * (N // R)] * tw[r * p * (N // (done * R))][:, None] for r in range(R)])
        v = np.einsum('kr,rjn->kjn', _small(R, c), v)
        y = np.empty_like(x)
        for r in range(R):
            y[(j // done) * done * R + p + r * done] = v[r]
        x, done = y, done * R
    return x * np.exp(2j * np.pi * (np.outer(k, n) % N) / N) - 1.0


def _summary(g):
    per_output = g.mean(1)
    return abs(g.mean()), np.sqrt(np.mean(np.abs(g) ** 2)), np.abs(per_output).max()


@pytest.mark.parametrize("plan", PLANS, ids=lambda p: '.'.join(map(str, p)))
def test_radix_16_constant(plan):
    c1, c2, t = _constants()
    nearest = float(f32(np.cos(np.pi / 8)))
    own, near = _summary(_gain_error(plan, (c1, c2, t))), _summary(_gain_error(plan, (nearest, c2, t)))
    print('.'.join(map(str, plan)), 'mean %.1e rms %.1e largest output %.1e, nearest %.1e %.1e %.1e' % (own + near))
    assert all(a <= b for a, b in zip(own, near))
    # the nearest constant's mean gain is 1 - 2.8e-8 to 1 - 4.7e-8
    assert own[0] <= 2e-8
