"""Factorisation kernels by front shape (lu_kernels.hip) against the systems
themselves: fronts around the widths where their parts can go wrong.

A system is `groups` sets of `k` unknowns, each coupled to the whole of one
dense block of `u` unknowns: the first sets become fronts of k + u rows with k
pivots, the last joins the dense block's panels (64 pivots, nested).  The
values are 6 I plus normal entries over the square root of the dimension, with
a positive definite symmetric part, so that elimination without pivoting stays
bounded and every l u term is of the size of the entries it changes.
"""

from __future__ import annotations

import numpy as np
import pytest
import scipy.sparse as sp

from test_gpu_lu_capi import _batch_values, _run

pytestmark = pytest.mark.gpu


def _system(groups, k, u, seed):
    n = groups * k + u
    M = np.zeros((n, n), bool)
    M[:, groups * k:] = M[groups * k:, :] = True
    for g in range(groups):
        M[g * k:(g + 1) * k, g * k:(g + 1) * k] = True
    v = np.random.default_rng(seed).standard_normal((n, n)) / np.sqrt(n) + 6.0 * np.eye(n)
    return sp.csr_matrix((v[M], np.nonzero(M)), shape=(n, n))


# ||x|| <= ||b|| / 2 (the symmetric part is at least 2) and || |L||U| || is at
# most sqrt(n) ||A||, ||A|| <= 9, so the residual stays below 4.5 n times the
# arithmetic's unit: 2^-53, 2^-24, and for the 3xBF16 products 2^-16 of their
# share, which adds as sqrt(n) 4.5 * 2^-16 at the most
BOUND = {0: lambda n: 4.5 * n * 2.0 ** -53, 1: lambda n: 4.5 * n * 2.0 ** -24,
         2: lambda n: 4.5 * n * 2.0 ** -24 + 4.5 * np.sqrt(n) * 2.0 ** -16}


# lane-per-scenario fronts of 9, 12, 13 and 16 rows (past the one-workgroup
# batch limit); fronts with 1, 3, 7, 17, 31, 32, 33 and 63 pivots on either
# side of a run of operands, of a lane group's share and of 32 pivots, beside
# contribution blocks one short of, at and past 64-column tiles; FP32 row
# blocks up to 512 rows and tiles past them
@pytest.mark.parametrize("groups,k,u,B", [
    (2, 1, 8, 2049), (3, 4, 8, 2049), (2, 5, 8, 2049), (2, 4, 12, 2049),
    (2, 1, 129, 3), (2, 3, 128, 65), (3, 7, 193, 2), (2, 17, 200, 3), (2, 31, 127, 5),
    (2, 32, 140, 3), (2, 33, 135, 3), (2, 63, 191, 2), (2, 3, 508, 2), (2, 5, 510, 2), (2, 35, 517, 2)])
@pytest.mark.parametrize("precision", [0, 1, 2])
def test_fronts(gpu, groups, k, u, B, precision):
    print(f"[fronts] {groups} x {k} + {u}, batch {B}, precision {precision}", flush=True)
    A = _system(groups, k, u, 1000 * k + u)
    n = A.shape[0]
    vals = _batch_values(A, B, 3)
    rhs = np.random.default_rng(4).standard_normal((B, n))
    x, xt, flags, _ = _run(gpu, A, vals, rhs, precision, 64, 0)
    assert not flags.any()
    for b in np.unique(np.r_[np.arange(min(B, 70)), B - 1]):
        M = sp.csr_matrix((vals[b], A.indices, A.indptr), shape=A.shape)
        for r in (M @ x[b] - rhs[b], M.T @ xt[b] - rhs[b]):
            assert np.linalg.norm(r) <= BOUND[precision](n) * np.linalg.norm(rhs[b]), b
