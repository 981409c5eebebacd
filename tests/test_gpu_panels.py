"""Systems of orders above 128 (wide panels): the edges of the 64-row lanes, of the 256-row
blocks of the residual and of the panels, against the CPU oracle."""
import numpy as np
import pytest

import oracle
from staccato_amd import synth

pytestmark = pytest.mark.gpu

EDGES = [129, 143, 145, 160, 191, 193, 255, 256, 257, 272, 321, 385, 511, 512, 513, 703, 1024]


def _check(handle, ops, n, rhs, seed):
    rom, rng = synth.modal_rom(n, seed, 0.02, alpha=1e-4, beta=0.5)
    K, M, D = rom.K, rom.M, rom.D
    if ops == "undamped":
        D = None
    elif ops == "complex":
        K, M, D = (a * (1 + 1e-3j) for a in (K, M, D))
    handle.rom_set(0, K, M, D, rom.eta)
    freq = np.array([3.0, 410.0, 1300.0])
    kappa = synth.cond2(rom, freq).max()
    # LU with partial pivoting and no growth: n u; the refinement stops at 1e-14
    back = {"plain": max(1e-14, n * 2.2e-16), "refined": 1e-14}
    for nrhs in rhs:
        F = synth.complex_normal(rng, (n, nrhs))
        Xo, io, _, _ = oracle.sweep(K, M, D, rom.eta, freq, F)
        assert (io == 0).all()
        for mode in ("plain", "refined"):
            X, info, be, _ = handle.sweep(0, freq, F, mode=mode, tol=1e-14)
            assert (info == 0).all()
            assert be.max() <= back[mode], (nrhs, mode)
            # forward error: kappa times the backward errors of both sides, the infinity
            # norms within sqrt(n) of the 2-norm
            err = np.abs(X - Xo).max() / np.abs(Xo).max()
            assert err <= (back[mode] + back["plain"]) * kappa * np.sqrt(n) + 1e-14, (nrhs, mode)


@pytest.mark.parametrize("n", EDGES)
def test_sweep_at_edges(handle, n):
    _check(handle, "rayleigh", n, (1, 5), 400 + n)


@pytest.mark.parametrize("ops", ["undamped", "complex"])
@pytest.mark.parametrize("n", [130, 256, 300, 520])
def test_operator_kinds(handle, ops, n):
    _check(handle, ops, n, (2, 3), 700 + n)
