"""Bounds of the simplex noise that the block sampling rests on: |n| < 1 (so
that its clamp never acts and it is twice differentiable everywhere), and the
norms of its gradient and Hessian, over a simplex's positions and all
gradient choices at its corners.  The kernels' constants stay above them.
"""
import re
from pathlib import Path

import numpy as np

SOURCE = (Path(__file__).resolve().parent.parent / "binarymeshfitting_amd" / "csrc" / "bmf_kernels.hip").read_text()
G = np.array([(a, b, 0) for a in (1, -1) for b in (1, -1)] + [(a, 0, b) for a in (1, -1) for b in (1, -1)]
             + [(0, a, b) for a in (1, -1) for b in (1, -1)], float)
CORNERS = np.array([(0, 0, 0), (1, 0, 0), (1, 1, 0), (1, 1, 1)], float)
SCALE, R2 = 76.8, 0.5


def _corner_terms(p):
    """Value, gradient and Hessian of each corner's term for its 12 gradients."""
    vals, grads, hess = [], [], []
    for k in range(4):
        x = p - CORNERS[k] + k / 6.0
        t = max(R2 - x @ x, 0.0)
        L = G @ x
        xg = x[None, :, None] * G[:, None, :]
        vals.append(SCALE * t ** 4 * L)
        grads.append(SCALE * (t ** 4 * G - 8 * t ** 3 * L[:, None] * x))
        hess.append(SCALE * (-8 * t ** 3 * (xg + xg.transpose(0, 2, 1))
                             + L[:, None, None] * (-8 * t ** 3 * np.eye(3) + 48 * t * t * np.outer(x, x))))
    return vals, grads, hess


def _all_sums(parts):
    a, b, c, d = parts
    s = a[:, None, None, None] + b[None, :, None, None] + c[None, None, :, None] + d[None, None, None, :]
    return s.reshape((-1,) + a.shape[1:])


def _norm3(A):
    """Largest |eigenvalue| of symmetric 3x3 matrices (trigonometric form)."""
    q = np.trace(A, axis1=1, axis2=2) / 3
    p = np.sqrt(np.maximum(((A - q[:, None, None] * np.eye(3)) ** 2).sum((1, 2)) / 6, 1e-30))
    r = np.clip(np.linalg.det((A - q[:, None, None] * np.eye(3)) / p[:, None, None]) / 2, -1, 1)
    phi = np.arccos(r) / 3
    return np.maximum(abs(q + 2 * p * np.cos(phi)), abs(q + 2 * p * np.cos(phi + 2 * np.pi / 3)))


def test_noise_derivative_bounds():
    hess_bound = float(re.search(r"kNoiseHess = ([0-9.]+)f", SOURCE).group(1))
    V = CORNERS - np.arange(4)[:, None] / 6.0
    n = 8
    points = [np.array([a, b, c, n - a - b - c]) / n for a in range(n + 1) for b in range(n + 1 - a)
              for c in range(n + 1 - a - b)]
    points.append(np.array([0.67797362, 0.29792432, 0.01419632, 0.00990573]))  # where a search ends
    top = [0.0, 0.0, 0.0]
    for w in points:
        vals, grads, hess = _corner_terms(w @ V)
        top[0] = max(top[0], sum(np.abs(v).max() for v in vals))
        top[1] = max(top[1], sum(np.linalg.norm(g, axis=1).max() for g in grads))
        top[2] = max(top[2], _norm3(_all_sums(hess)).max())
    print(top)
    assert top[0] < 1.0
    assert top[1] < 7.1
    assert 48.0 < top[2] < hess_bound / 1.03
