"""Bounds of gridded cells, for the GPU tests of the stage gridding calls.

The tolerance of a cell is that of an FP32 sum in any order: a term of the
sum is rounded once, and m terms are added with m - 1 further roundings, so either
component lies within (m + 2) 2^-24 sum |v w| of the exact sum, with m and the sum over
the visibilities (or footprints) that reach that cell.
"""
import numpy as np

import oracle
from imager_amd import synth


def _round(x):
    return np.sign(x) * np.floor(np.abs(x) + 0.5)


def footprint_sums(o, n, K, with_sinc, value):
    """Per channel of timestep 0: number of footprint cells (K = 0: of nearest cells) and sum
    of |value * weight| in each cell, over the unflagged baselines."""
    table = np.abs(oracle.kb_kernels(K, with_sinc)) if K else None
    ok = (o.flags == 0) & np.isfinite(value).all(axis=0)
    terms = np.zeros((o.n_ch, n, n))
    sums = np.zeros((o.n_ch, n, n))
    for ch in range(o.n_ch):
        wl = synth.C_LIGHT / o.freq[ch]
        cells, rows = [], []
        for x, d in ((o.u, o.delta_u), (o.v, o.delta_v)):
            e = x.astype(np.float64)[ok] / wl / d
            p = _round(e)
            cells.append(p.astype(np.int64))
            rows.append((_round((e - p) * 1023.0).astype(np.int64) + 1534) % 1023)
        a = np.abs(value[ch][ok])
        for s in (1, -1):
            if not K:
                at = ((s * cells[1]) % n, (s * cells[0]) % n)
                np.add.at(terms[ch], at, 1.0)
                np.add.at(sums[ch], at, a)
            for j in range(K):
                for c in range(K):
                    at = []
                    for p, k in ((cells[0], c), (cells[1], j)):
                        i = s * (p - K // 2 + k) + n // 2
                        at.append(np.where(i < n // 2, i + n // 2, i - n // 2))
                    x, y = at
                    inside = (x >= 0) & (x < n) & (y >= 0) & (y < n)
                    w = a * table[rows[0], c] * table[rows[1], j]
                    np.add.at(terms[ch], (y[inside], x[inside]), 1.0)
                    np.add.at(sums[ch], (y[inside], x[inside]), w[inside])
    return terms, sums


def assert_within(got, want, terms, sums):
    """Both components of every cell within (terms + 2) 2^-24 sums, which has to be far below
    the values themselves."""
    bound = (terms + 2.0) * 2.0 ** -24 * sums
    assert bound.max() < 1e-2 * np.abs(want).max()
    d = got - want
    assert (np.abs(d.real) - bound).max() <= 0.0
    assert (np.abs(d.imag) - bound).max() <= 0.0


def undersampled(n_ant, n_ch, n, seed, reach=1.35):
    """Baselines whose cells lie anywhere within `reach` * N of the origin."""
    o = synth.small(n_ant=n_ant, n_ch=n_ch, n_t=1, n_pixels=n, seed=seed, bl_flag_fraction=0.2)
    rng = np.random.Generator(np.random.PCG64(seed))
    pos = rng.uniform(-reach, reach, (2, o.n_bl)) * n
    o.delta_u = o.delta_v = 1.0
    lam = synth.C_LIGHT / o.freq[0]
    o.u = (pos[0] * lam).astype(np.float32)
    o.v = (pos[1] * lam).astype(np.float32)
    return o
