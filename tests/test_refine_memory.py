"""Workspace of the refined solve: the residual's partials stay small beside the
matrices, and from n = 11,600 on are those of one group of 8 right-hand sides."""
import ctypes

import pytest


@pytest.mark.parametrize("nrhs", [1, 8, 9, 32, 100])
def test_residual_partials(bfa, nrhs):
    lib = bfa.lib()
    lib.bfa_refine_partials.restype = ctypes.c_size_t
    for n in (1, 64, 270, 1350, 5760, 8000, 11400, 11600, 20000, 60000):
        b = lib.bfa_refine_partials(n, nrhs)
        one = -(-n // 256) * min(nrhs, 8) * n * 16
        assert b >= one
        # complex128 matrix and complex64 factors: 24 n^2 bytes; the partials are
        # n^2 16 min(nrhs, 32) / 32 bytes where the chunks are shortest
        assert b <= max(24 * n * n, 16 * 32 * n)
        if n >= 5000:
            assert b <= 24 * n * n / 8 and b <= max(one, 150 << 20)
        if n >= 11600:
            assert b == one
