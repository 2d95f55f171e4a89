"""The segmented y-line sweeps (line_step in vfs_v3p2_amd/csrc/pp_line_dev.hpp):
both Thomas sweeps are affine recurrences, so a line split into S segments, each
swept from a zero carry with the product of its multipliers kept and chained through
the segments' carries, solves the same tridiagonal system as the sequential sweep.
`segmented` re-sweeps every segment from its carry; `affine`, the form the kernels
take, adds the carry times the row's running product.  Checked here in FP64 on
diagonally dominant systems of 1 to 256 rows for 16 and 32 segments, including lines
shorter than the segment count (empty segments carry the identity), and the affine
form's FP32 error against the sequential sweep's."""
import numpy as np
import pytest


def thomas_factors(a, b, c):
    ny = len(b)
    cp, inv = np.zeros(ny), np.zeros(ny)
    prev = 0.0
    for j in range(ny):
        den = b[j] - a[j] * prev
        inv[j] = 1.0 / den
        prev = c[j] * inv[j]
        cp[j] = prev
    return cp, inv


def sequential(a, cp, inv, r):
    ny = len(r)
    d = np.zeros(ny)
    dp = 0.0
    for j in range(ny):
        dp = (r[j] - a[j] * dp) * inv[j]
        d[j] = dp
    z = np.zeros(ny)
    zn = 0.0
    for j in range(ny - 1, -1, -1):
        zn = d[j] - cp[j] * zn
        z[j] = zn
    return z


def segmented(a, cp, inv, r, S):
    ny = len(r)
    L = (ny + S - 1) // S
    rows = [(s * L, max(0, min(L, ny - s * L))) for s in range(S)]
    part = np.zeros((2, S))
    for s, (j0, nr) in enumerate(rows):
        dl, pr = 0.0, 1.0
        for j in range(j0, j0 + nr):
            dl = (r[j] - a[j] * dl) * inv[j]
            pr = pr * -(a[j] * inv[j])
        part[:, s] = dl, pr
    carry, c = np.zeros(S), 0.0
    for t in range(S):
        carry[t] = c
        c = part[0, t] + part[1, t] * c
    d = np.zeros(ny)
    for s, (j0, nr) in enumerate(rows):
        dp = carry[s]
        for j in range(j0, j0 + nr):
            dp = (r[j] - a[j] * dp) * inv[j]
            d[j] = dp
    for s, (j0, nr) in enumerate(rows):
        zl, pr = 0.0, 1.0
        for j in range(j0 + nr - 1, j0 - 1, -1):
            zl = d[j] - cp[j] * zl
            pr = pr * -cp[j]
        part[:, s] = zl, pr
    c = 0.0
    for t in range(S - 1, -1, -1):
        carry[t] = c
        c = part[0, t] + part[1, t] * c
    z = np.zeros(ny)
    for s, (j0, nr) in enumerate(rows):
        zn = carry[s]
        for j in range(j0 + nr - 1, j0 - 1, -1):
            zn = d[j] - cp[j] * zn
            z[j] = zn
    return z


@pytest.mark.parametrize("segs", [16, 32])
@pytest.mark.parametrize("ny", [1, 5, 16, 17, 31, 100, 128, 255, 256])
def test_segmented_sweeps_solve_the_line(ny, segs):
    rng = np.random.default_rng(ny + 1000 * segs)
    a = rng.uniform(-1.0, 0.0, ny)
    c = rng.uniform(-1.0, 0.0, ny)
    b = 2.5 + rng.uniform(0.0, 1.0, ny)
    a[0] = 0.0
    c[-1] = 0.0
    if ny > 8:
        # a cell without an unknown: identity row, as the factors store it
        a[3], b[3], c[3] = 0.0, 1.0, 0.0
    cp, inv = thomas_factors(a, b, c)
    r = rng.standard_normal(ny)
    z_seq = sequential(a, cp, inv, r)
    z_seg = segmented(a, cp, inv, r, segs)
    T = np.diag(b) + np.diag(a[1:], -1) + np.diag(c[:-1], 1)
    assert np.abs(T @ z_seg - r).max() <= 1e-14 * max(1.0, np.abs(r).max())
    assert np.abs(z_seg - z_seq).max() <= 1e-14 * np.abs(z_seq).max()


def affine(a, cp, inv, r, S, dt=np.float64):
    a, cp, inv, r = (v.astype(dt) for v in (a, cp, inv, r))
    ny = len(r)
    L = (ny + S - 1) // S
    rows = [range(s * L, s * L + max(0, min(L, ny - s * L))) for s in range(S)]
    d, P = np.zeros(ny, dt), np.zeros(ny, dt)
    ends = []
    for seg in rows:
        v, p = dt(0), dt(1)
        for j in seg:
            v, p = dt((r[j] - a[j] * v) * inv[j]), dt(p * -(a[j] * inv[j]))
            d[j], P[j] = v, p
        ends.append((v, p))
    c, up = dt(0), np.zeros(ny, dt)
    for seg, (v, p) in zip(rows, ends):
        for j in seg:
            up[j] = d[j] + P[j] * c
        c = dt(v + p * c)
    ends = []
    for seg in rows:
        v, p = dt(0), dt(1)
        for j in reversed(seg):
            v, p = dt(up[j] - cp[j] * v), dt(p * -cp[j])
            d[j], P[j] = v, p
        ends.append((v, p))
    c, z = dt(0), np.zeros(ny, dt)
    for seg, (v, p) in reversed(list(zip(rows, ends))):
        for j in seg:
            z[j] = d[j] + P[j] * c
        c = dt(v + p * c)
    return z


@pytest.mark.parametrize("segs", [16, 32])
@pytest.mark.parametrize("ny", [1, 5, 16, 17, 31, 100, 128, 255, 256])
def test_affine_sweeps_solve_the_line(ny, segs):
    rng = np.random.default_rng(ny + 1000 * segs)
    a, c = rng.uniform(-1.0, 0.0, (2, ny))
    b = 2.05 + rng.uniform(0.0, 0.1, ny)
    a[0] = c[-1] = 0.0
    if ny > 8:
        a[3], b[3], c[3] = 0.0, 1.0, 0.0
    cp, inv = thomas_factors(a, b, c)
    r = rng.standard_normal(ny)
    z_seq = sequential(a, cp, inv, r)
    scale = np.abs(z_seq).max()
    assert np.abs(affine(a, cp, inv, r, segs) - z_seq).max() <= 1e-14 * scale
    # in FP32 every value sees at most one more rounding of a product and a sum per sweep
    # than in the sequential sweep, whose own error is a few eps on these systems
    f = np.float32
    e_seq = np.abs(affine(a, cp, inv, r, 1, f) - z_seq).max() / scale  # one segment: the sequential sweep
    e_aff = np.abs(affine(a, cp, inv, r, segs, f) - z_seq).max() / scale
    assert e_aff <= e_seq + 4 * np.finfo(f).eps
