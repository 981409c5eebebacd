"""Ends of the floating-point range: entries of A(w) and solutions that overflow stay with the
degrees of freedom they belong to."""
import numpy as np
import pytest

from staccato_amd import synth

pytestmark = pytest.mark.gpu

# every factorisation: registers (the column groups), wide panels of one and two workgroups
# per CU, the register panel
ORDERS = [5, 33, 64, 80, 128, 129, 200, 257, 513]


@pytest.mark.parametrize("at", [0, 2])
@pytest.mark.parametrize("n", ORDERS)
def test_overflowing_mass_holds_its_dof(handle, n, at):
    """A(w) has an infinite diagonal entry: that unknown is zero, the others solve the system
    without it.  at = 0: a coupled degree of freedom (its pivot is the first); 2: an
    uncoupled one further on (its row can be no earlier column's pivot)."""
    rom, rng = synth.modal_rom(n, 300 + n, 0.02)
    K, M = rom.K.copy(), rom.M.copy()
    if at:
        K[at, :] = K[:, at] = M[at, :] = M[:, at] = 0.0
    M[at, at] = 1e305
    freq = np.array([40.0, 410.0])
    F = synth.complex_normal(rng, (n, 3))
    handle.rom_set(0, K, M, None, rom.eta)
    X, info, _, _ = handle.sweep(0, freq, F, mode="plain", berr=False)
    assert (info == 0).all()
    keep = np.arange(n) != at
    for j, f in enumerate(freq):
        A = ((1 + 1j * rom.eta) * K - (2 * np.pi * f) ** 2 * np.where(M > 1e300, 0.0, M))[np.ix_(keep, keep)]
        ref = np.linalg.solve(A, F[keep])
        assert (X[j, at] == 0).all()
        # LU with partial pivoting on both sides: n u each, times the condition number
        tol = 2 * n * 2.2e-16 * np.linalg.cond(A) * np.sqrt(n) + 1e-14
        assert np.abs(X[j, keep] - ref).max() <= tol * np.abs(ref).max()


@pytest.mark.parametrize("n", [1, 5, 33, 64, 65, 100, 128, 129, 300])
def test_overflowing_unknown_leaves_the_others(handle, n):
    """The first unknown of a diagonal system, found last, overflows: not finite, and the only one."""
    d = np.full(n, 2.0 + 0j)
    d[0] = 1e-10
    B = np.full((n, 2), 1.0 + 0j)
    B[0, 1] = 1e305
    X, info, _, _ = handle.gesv_batched(np.diag(d)[None], B, mode="plain", berr=False)
    assert list(info) == [0]
    ref = np.full((n, 2), 0.5 + 0j)
    ref[0] = 1e10
    assert not np.isfinite(X[0, 0, 1])
    X[0, 0, 1] = ref[0, 1]
    # one division each: two roundings
    np.testing.assert_allclose(X[0], ref, rtol=1e-15, atol=0)


@pytest.mark.parametrize("n,mode,kernel,budget", [(143, "refined", 1, 16384), (230, "refined", 1, 20480),
                                                  (74, "refined", 2, 16384), (843, "refined", 2, 120000),
                                                  (29, "plain", 1, 16384), (270, "plain", 1, 32768),
                                                  (400, "plain", 2, 110000)])
def test_smallest_lds_budgets(handle, n, mode, kernel, budget):
    rom, rng = synth.modal_rom(n, 40 + n, 0.02)
    F = synth.complex_normal(rng, (n, 2))
    handle.rom_set(0, rom.K, rom.M, rom.D, rom.eta)
    try:
        handle.set_policy(n, mode, kernel, budget, 0)
        _, info, be, _ = handle.sweep(0, [40.0, 410.0, 1300.0], F, mode=mode, tol=1e-12)
    finally:
        handle.clear_policies()
    assert (info == 0).all() and be.max() <= 1e-12


@pytest.mark.parametrize("at", [0, 20, 40, 100])
@pytest.mark.parametrize("n", [129, 144, 200, 256, 300])
def test_mass_beyond_complex64(handle, n, at):
    """Refined, an uncoupled mass whose diagonal entry overflows in complex64 only: its pivot
    is infinite, the other unknowns are those of the system without it.  The norm of A(w)
    makes any solution meet the tolerance, so they are as good as the complex64 factors."""
    rom, rng = synth.modal_rom(n, 700 + n, 0.02)
    K, M = rom.K.copy(), rom.M.copy()
    K[at, :] = K[:, at] = M[at, :] = M[:, at] = 0.0
    M[at, at] = 1e45
    freq = np.array([40.0, 410.0])
    F = synth.complex_normal(rng, (n, 2))
    handle.rom_set(0, K, M, None, rom.eta)
    X, info, be, _ = handle.sweep(0, freq, F, mode="refined", tol=1e-10)
    assert (info == 0).all() and be.max() <= 1e-10
    keep = np.arange(n) != at
    for j, f in enumerate(freq):
        A = ((1 + 1j * rom.eta) * K - (2 * np.pi * f) ** 2 * M)[np.ix_(keep, keep)]
        ref = np.linalg.solve(A, F[keep])
        assert np.abs(X[j, at]).max() <= 1e-40
        # backward error of the factors and solves: at most n u in complex64
        tol = n * 2.0 ** -24 * np.linalg.cond(A) * np.sqrt(n)
        assert np.abs(X[j, keep] - ref).max() <= tol * np.abs(ref).max()
