"""Systems solved in registers (orders up to 128): the edges of the 64-row lanes, of the
four-column blocks and of the column groups, against the CPU oracle."""
import numpy as np
import pytest

import oracle
from staccato_amd import synth

pytestmark = pytest.mark.gpu

EDGES = [1, 3, 4, 5, 31, 32, 33, 63, 64, 65, 95, 96, 97, 127, 128]


def _rel(a, b):
    return np.abs(a - b).max() / np.abs(b).max()


@pytest.mark.parametrize("n", EDGES)
def test_sweep_at_edges(handle, n):
    """Both modes; 1 right-hand side, and 9 (a second factorisation or group)."""
    rom, rng = synth.modal_rom(n, 900 + n, 0.02, alpha=1e-4, beta=0.5)
    handle.rom_set(0, rom.K, rom.M, rom.D, rom.eta)
    freq = np.array([1.0, 77.0, 500.0, 1300.0])
    kappa = synth.cond2(rom, freq).max()
    for nrhs in (1, 9):
        F = synth.complex_normal(rng, (n, nrhs))
        Xo, io, _, _ = oracle.sweep(rom.K, rom.M, rom.D, rom.eta, freq, F)
        assert (io == 0).all()
        for mode, tol in (("plain", 1e-14), ("refined", 1e-14)):
            X, info, be, st = handle.sweep(0, freq, F, mode=mode, tol=1e-14)
            assert (info == 0).all()
            assert be.max() <= tol
            # backward errors of 1e-14 on both sides: forward error kappa times that, the
            # infinity norms within sqrt(n) of the 2-norm
            assert _rel(X, Xo) <= 2e-14 * kappa * np.sqrt(n) + 1e-14, (nrhs, mode)


@pytest.mark.parametrize("n", [2, 17, 64, 66, 128])
def test_adjoint_at_edges(handle, n):
    rom, rng = synth.modal_rom(n, 950 + n, 0.02)
    F = synth.complex_normal(rng, (n, 3))
    c = synth.complex_normal(rng, (n,))
    freq = np.linspace(5.0, 900.0, 7)
    handle.rom_set(0, rom.K, rom.M, rom.D, rom.eta)
    J, ds, de, info = handle.adjoint(0, freq, F, c, rom.Phi, rom.kdiag)
    Jc, dsc, dec = synth.adjoint_closed_form(rom, freq, F, c)
    assert (info == 0).all()
    # the closed form itself is good to kappa u (as for the larger adjoint tests)
    tol = 1e-8
    assert abs(J / Jc - 1) < tol and abs(de / dec - 1) < tol
    assert np.abs(ds - dsc).max() <= tol * np.abs(dsc).max()


@pytest.mark.parametrize("mode", ["plain", "refined"])
def test_pivots_ties_and_zeros(handle, mode):
    """Explicit matrices whose pivot search meets ties, zero columns to the pivot's
    left, entries far from 1 and a singular matrix; the batch's other members are unharmed."""
    rng = np.random.default_rng(5)
    n = 40
    A = synth.complex_normal(rng, (6, n, n))
    A[0] = np.fft.fft(np.eye(n)) / np.sqrt(n)               # magnitudes tie up to rounding
    A[1] = np.eye(n)[rng.permutation(n)]                    # a permutation: zeros and exact ties
    A[2] *= 1e200 if mode == "plain" else 1e15
    A[3] *= 1e-200 if mode == "plain" else 1e-15
    A[4][:, 7] = 0.0                                        # singular at column 8
    B = synth.complex_normal(rng, (n, 2))
    X, info, be, _ = handle.gesv_batched(A, B, mode=mode, tol=1e-12)
    assert list(info) == [0, 0, 0, 0, 8, 0]
    assert np.isnan(X[4]).all()
    for j in (0, 1, 2, 3, 5):
        ref = np.linalg.solve(A[j], B)
        assert be[j].max() <= 1e-12
        assert _rel(X[j], ref) <= 1e-11 * np.linalg.cond(A[j])
