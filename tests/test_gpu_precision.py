"""Rounding errors of the complex64 factorisation and solves, against LAPACK's in complex64."""
import numpy as np
import pytest
import scipy.linalg as sl

from staccato_amd import synth

pytestmark = pytest.mark.gpu

FREQ = np.array([2.0, 77.0, 310.0, 650.0, 990.0, 1500.0])


def _factor_error(A, LU, ipiv):
    """|| P A - L U || / || A ||, the products in 64 bits."""
    n = A.shape[0]
    perm = np.arange(n)
    for i, q in enumerate(ipiv):
        perm[[i, q]] = perm[[q, i]]
    L, U = np.tril(LU, -1).astype(np.complex128) + np.eye(n), np.triu(LU).astype(np.complex128)
    A = A.astype(np.complex128)
    return np.linalg.norm(A[perm] - L @ U) / np.linalg.norm(A)


@pytest.mark.parametrize("n", [192, 256])
def test_factor_error(handle, n):
    """Mean over 24 matrices.  Gauss's three products converted every 32 columns measured 2.14
    to 2.15 times LAPACK's error (72 matrices), as right-looking panels of that width; with
    the three sums kept over all finished columns 2.22 to 2.29."""
    e, el = [], []
    for seed in range(2):
        for damping in ({}, dict(alpha=1e-4, beta=0.5)):
            rom, _ = synth.modal_rom(n, 100 * n + seed, 0.02, **damping)
            handle.rom_set(0, rom.K, rom.M, rom.D, rom.eta)
            LU, ipiv, info = handle.getrf(0, FREQ, mode="refined")
            assert (info == 0).all()
            for j, f in enumerate(FREQ):
                A = synth.assemble(rom, f).astype(np.complex64)
                e.append(_factor_error(A, LU[j], ipiv[j] - 1))
                el.append(_factor_error(A, *sl.lu_factor(A)))
    assert np.mean(e) <= 2.18 * np.mean(el), (np.mean(e), np.mean(el))


@pytest.mark.parametrize("n", [320, 512, 1024])
def test_first_solve_sums(handle, n):
    """Unrefined solution (tol = 1) of a unit upper triangular system of equal entries c, all
    unknowns 1: the i-th row from below subtracts c from b_i = 1 + c i, i times.  Summed in blocks of 16
    first, the n / 16 subtractions round by u times a partial sum that falls from c i to 0,
    n / 64 u of the backward error's denominator 2 c n, the sums within the blocks by 4.3 u,
    the rounded load by half a u, the block's inverse by less than 2 u."""
    c = float(np.float32(0.37))
    A = np.triu(np.full((n, n), c + 0j), 1) + np.eye(n)
    b = A @ np.ones((n, 1))
    _, info, be, _ = handle.gesv_batched(A[None], b, mode="refined", tol=1.0)
    assert info[0] == 0
    assert be[0, 0] <= (n / 64 + 7) * 2.0 ** -24, be[0, 0] * 2.0 ** 24
