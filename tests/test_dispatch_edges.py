"""Edges of the kernel selection on the CPU (configurations, generated sources, emulator): what
a general path accepts and computes, a faster path accepts and computes as well."""
import numpy as np
import pytest

import bbfft_amd as bb
from emu import runner

PER_TILE_IDS, MATRIX = 512, 2048


def _cfg(M, N, K, fp, d, t, istride=None, ostride=None):
    cfg = bb.configuration(1, [M, N, K], bb.precision(fp), bb.direction(d),
                           bb.transform_type(t))
    cfg.set_strides_default(False)
    if istride:
        cfg.istride = istride
    if ostride:
        cfg.ostride = ostride
    return cfg


@pytest.mark.parametrize("bad", [np.inf, np.nan])
@pytest.mark.parametrize("fp", [4, 8])
@pytest.mark.parametrize("M,N,fac,Nt,Kb", [(1, 37, [37], 16, 4), (2, 61, [61], 32, 1),
                                           (1, 74, [37, 2], 32, 2)])
def test_matrix_sums_of_values_that_are_not_finite(M, N, fac, Nt, Kb, fp, bad):
    """One infinite or NaN input: the matrix products leave the same outputs infinite and NaN,
    component by component, as the butterfly in registers does."""
    K = 3
    for d in (-1, 1):
        for at in (0, 1, N - 2):
            x = np.ones((K, N, M), np.complex64 if fp == 4 else np.complex128)
            x[1, at, M - 1] = bad
            cfg = _cfg(M, N, K, fp, d, 0)
            y = [runner.run(bb, cfg, x.ravel(), x.size, tuning=dict(
                factorization=fac, Nt=Nt, Mb=M, Kb=Kb, no_pad=True, flags=f))
                for f in (PER_TILE_IDS, PER_TILE_IDS | MATRIX)]
            for part in (np.real, np.imag):
                assert np.array_equal(np.isnan(part(y[0])), np.isnan(part(y[1]))), (d, at)
                assert np.array_equal(np.isinf(part(y[0])), np.isinf(part(y[1]))), (d, at)
