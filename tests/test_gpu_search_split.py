# -*- coding: utf-8 -*-
"""Index search on split products: ragged row and query counts, and values
outside fp16's range."""

from __future__ import annotations

import numpy as np
import pytest

from rvc_hip.pipeline import HipVcGlue

pytestmark = pytest.mark.gpu


def _case(N, F, D, seed):
    r = np.random.default_rng(seed)
    v = r.standard_normal((N, D), dtype=np.float32)
    q = 0.8 * v[r.integers(0, N, F)] + 0.4 * r.standard_normal((F, D), dtype=np.float32)
    return v, q.astype(np.float32)


def _search(v, q):
    glue = HipVcGlue()
    glue.set_index(v)
    return glue.search(q)


@pytest.mark.parametrize("N,F,D", [(9, 1, 320), (127, 31, 768), (129, 33, 768), (1000, 65, 1024)])
def test_rows_and_distances(N, F, D):
    v, q = _case(N, F, D, N + F)
    scores, rows = _search(v, q)
    d = ((q[:, None].astype(np.float64) - v[None].astype(np.float64)) ** 2).sum(-1)
    want = np.sort(d, axis=1)[:, :scores.shape[1]]
    # |q|^2 + |v|^2 - 2 q v: sums of D products, each about 2^-24 of |q|^2 + |v|^2
    size = (q.astype(np.float64) ** 2).sum(1)[:, None] + (v.astype(np.float64) ** 2).sum(1).max()
    assert (np.abs(scores - want) <= 2e-6 * size).all()
    assert (np.abs(np.take_along_axis(d, rows, 1) - want) <= 4e-6 * size).all()


@pytest.mark.parametrize("exponent", [-40, -12, 12, 40])
def test_scale_of_the_values(exponent):
    v, q = _case(300, 40, 768, 5)
    s = np.float32(2.0) ** exponent
    scores, rows = _search(v, q)
    got, at = _search(v * s, q * s)
    assert (at == rows).mean() > 0.998
    # distances scale by the power of two squared, up to the sums' rounding
    size = (q ** 2).sum(1)[:, None] + (v ** 2).sum(1).max()
    assert (np.abs(got / s / s - scores) <= 2e-6 * size).all()


def test_infinite_and_nan_rows_are_never_found():
    v, q = _case(300, 40, 768, 6)
    w = v.copy()
    w[17, 3], w[50, 4] = np.nan, np.inf
    scores, rows = _search(w, q)
    assert np.isfinite(scores).all() and not np.isin(rows, (17, 50)).any()


@pytest.mark.parametrize("exponent", [-60, -20, 12, 20, 60])
def test_a_query_does_not_hang_on_its_neighbours(exponent):
    """Queries of another size, an infinite and a NaN one share tiles with the
    rest, whose distances stay bit for bit what they are without them."""
    v, q = _case(300, 70, 768, 7)
    scores, rows = _search(v, q)
    other = q.copy()
    other[5::16] *= np.float32(2.0) ** exponent
    other[9, 3], other[41, 700] = np.nan, np.inf
    keep = np.ones(len(q), bool)
    keep[5::16] = keep[[9, 41]] = False
    got, at = _search(v, other)
    np.testing.assert_array_equal(got[keep], scores[keep])
    np.testing.assert_array_equal(at[keep], rows[keep])
