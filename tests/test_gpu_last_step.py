"""Wide panels whose last step has room for the right-hand sides, and those just without: sizes
around the step (16 columns complex128, 32 complex64), one and two panels a step."""
import numpy as np
import pytest

import oracle
from staccato_amd import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [129, 140, 141, 143, 156, 157, 159, 160, 268, 269, 300, 541])
@pytest.mark.parametrize("jb", [0, 16])
def test_sweep_and_explicit(handle, n, jb):
    rom, rng = synth.modal_rom(n, 60 + n, 0.02, alpha=1e-4, beta=0.5)
    freq = np.array([3.0, 700.0])
    A = np.stack([synth.assemble(rom, f) for f in freq])
    kappa = synth.cond2(rom, freq).max()
    handle.rom_set(0, rom.K, rom.M, rom.D, rom.eta)
    try:
        for mode in ("plain", "refined"):
            if jb:
                handle.set_policy(n, mode, 2, 0, jb)
            # LU with partial pivoting and no growth: n u; the refinement stops at 1e-14
            back = max(1e-14, n * 2.2e-16) if mode == "plain" else 1e-14
            for nrhs in (1, 3, 4, 5):
                F = synth.complex_normal(rng, (n, nrhs))
                Xo, io, _, _ = oracle.sweep(rom.K, rom.M, rom.D, rom.eta, freq, F)
                assert (io == 0).all()
                for X, info, be, _ in (handle.sweep(0, freq, F, mode=mode, tol=1e-14),
                                       handle.gesv_batched(A, F, mode=mode, tol=1e-14)):
                    assert (info == 0).all() and be.max() <= back, (mode, nrhs)
                    # the backward errors of both sides times kappa, infinity norms within sqrt(n)
                    err = np.abs(X - Xo).max() / np.abs(Xo).max()
                    assert err <= 2 * back * kappa * np.sqrt(n) + 1e-14, (mode, nrhs)
    finally:
        handle.clear_policies()


def test_a_narrow_last_step_costs_little(handle):
    """n = 129, plain, one load: 0.88 of the time of n = 144 (nine full steps); with a pass of
    its own for the load after the step of one column 0.94."""
    import time
    import torch
    calls, keep = [], []
    st = torch.cuda.Stream()
    for rid, n in enumerate((129, 144)):
        rom, rng = synth.modal_rom(n, n, 0.02)
        handle.rom_set(rid, rom.K, rom.M, None, rom.eta)
        f_t = torch.linspace(1.0, 1200.0, 1024, dtype=torch.float64, device="cuda")
        F_t = torch.from_numpy(synth.complex_normal(rng, (1, n))).cuda()
        X = torch.empty((1024, 1, n), dtype=torch.complex128, device="cuda")
        info = torch.empty(1024, dtype=torch.int32, device="cuda")
        keep.append((f_t, F_t, X, info))
        calls.append(lambda rid=rid, f=f_t, F=F_t, X=X, i=info: handle.sweep_dev(rid, f, F, X, i, stream=st.cuda_stream))
    torch.cuda.synchronize()
    best = [1e9, 1e9]
    for _ in range(8):
        for i, f in enumerate(calls):
            t = time.perf_counter()
            for _ in range(3):
                f()
            torch.cuda.synchronize()
            best[i] = min(best[i], time.perf_counter() - t)
    assert all((k[3] == 0).all() for k in keep)
    assert best[0] <= 0.91 * best[1], best[0] / best[1]
