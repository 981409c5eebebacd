"""The register kernel from the work queue (batches and plans whose orders are all at most 128,
several lane and column classes in one launch), repeated factorisations of the
eight-wavefront form, the adjoint over several of them, and complex operators."""
import numpy as np
import pytest

import oracle
from staccato_amd import Plan, synth
from staccato_amd._lib import SysDesc

pytestmark = pytest.mark.gpu

SIZES = [20, 33, 64, 65, 96, 128, 5, 47]


def _systems(handle, sizes, first=0):
    out = []
    for i, n in enumerate(sizes):
        rom, rng = synth.modal_rom(n, 800 + 10 * first + i, 0.02, alpha=1e-4, beta=0.5 * (i % 2))
        handle.rom_set(i, rom.K, rom.M, rom.D, rom.eta)
        freq = np.linspace(3.0, 1300.0, 3 + i)
        F = synth.complex_normal(rng, (n, 1 + (3 * i) % 10))
        Xo, io, _, _ = oracle.sweep(rom.K, rom.M, rom.D, rom.eta, freq, F)
        assert (io == 0).all()
        # backward errors of 1e-14 on both sides, the infinity norms within sqrt(n) of the 2-norm
        tol = 2e-14 * synth.cond2(rom, freq).max() * np.sqrt(n) + 1e-14
        out.append((freq, F, Xo, tol))
    return out


@pytest.mark.parametrize("mode", ["plain", "refined"])
@pytest.mark.parametrize("sizes", [SIZES, [8, 20, 31, 64], [128, 97]])
def test_batch(handle, mode, sizes):
    ss = _systems(handle, sizes)
    res, st = handle.sweep_batch([(i, f, F) for i, (f, F, _, _) in enumerate(ss)], mode=mode, tol=1e-14)
    for (f, F, Xo, tol), (X, info, be) in zip(ss, res):
        assert (info == 0).all() and be.max() <= 1e-14
        assert np.abs(X - Xo).max() <= tol * np.abs(Xo).max()
    assert st.points == sum(f.size for f, _, _, _ in ss)


@pytest.mark.parametrize("mode", ["plain", "refined"])
def test_plan(handle, mode):
    """Replayed with other loads in the same buffers, eager work in between."""
    import torch
    ss = _systems(handle, SIZES, first=1)
    keep, descs = [], (SysDesc * len(ss))()
    for i, (freq, F, _, _) in enumerate(ss):
        n, nrhs = F.shape
        t = (torch.from_numpy(freq).cuda(), torch.zeros((nrhs, n), dtype=torch.complex128, device="cuda"),
             torch.zeros((freq.size, nrhs, n), dtype=torch.complex128, device="cuda"),
             torch.full((freq.size,), 7, dtype=torch.int32, device="cuda"),
             torch.zeros((freq.size, nrhs), dtype=torch.float64, device="cuda"))
        keep.append(t)
        d = descs[i]
        d.rom_id, d.nfreq, d.freq_hz, d.nrhs = i, freq.size, t[0].data_ptr(), nrhs
        d.F, d.ldf, d.X, d.ldx, d.info, d.berr = t[1].data_ptr(), n, t[2].data_ptr(), n, t[3].data_ptr(), t[4].data_ptr()
    st = torch.cuda.Stream()
    torch.cuda.synchronize()
    plan = Plan(handle, descs, mode=mode, tol=1e-14)
    try:
        for rep in range(3):
            for t, (_, F, _, _) in zip(keep, ss):
                t[1].copy_(torch.from_numpy(np.ascontiguousarray(F.T)) * (rep + 1))
                t[2].zero_()
                t[3].fill_(7)
            torch.cuda.synchronize()
            plan.execute(st.cuda_stream)
            torch.cuda.synchronize()
            for t, (_, F, Xo, tol) in zip(keep, ss):
                X = t[2].cpu().numpy().transpose(0, 2, 1) / (rep + 1)
                assert (t[3].cpu().numpy() == 0).all() and t[4].max().item() <= 1e-14
                assert np.abs(X - Xo).max() <= tol * np.abs(Xo).max()
    finally:
        plan.close()


@pytest.mark.parametrize("n,nrhs", [(40, 9), (64, 17), (70, 16), (70, 17), (128, 17), (128, 33)])
def test_repeated_factorisations(handle, n, nrhs):
    """Few points, so that the register kernel is the choice whatever the loads."""
    rom, rng = synth.modal_rom(n, 70 + n, 0.02)
    handle.rom_set(0, rom.K, rom.M, None, rom.eta)
    freq = np.array([9.0, 870.0])
    F = synth.complex_normal(rng, (n, nrhs))
    Xo, _, _, _ = oracle.sweep(rom.K, rom.M, None, rom.eta, freq, F)
    tol = 2e-14 * synth.cond2(rom, freq).max() * np.sqrt(n) + 1e-14
    X, info, be, _ = handle.sweep(0, freq, F, mode="plain")
    assert (info == 0).all() and be.max() <= 1e-14
    assert np.abs(X - Xo).max() <= tol * np.abs(Xo).max()
    # the adjoint sums J and xi over the factorisations
    c = synth.complex_normal(rng, (n,))
    J, ds, de, info = handle.adjoint(0, freq, F, c, rom.Phi, rom.kdiag)
    Jc, dsc, dec = synth.adjoint_closed_form(rom, freq, F, c)
    assert (info == 0).all()
    # the closed form itself is good to kappa u (as for the other adjoint tests)
    assert abs(J / Jc - 1) < 1e-8 and abs(de / dec - 1) < 1e-8
    assert np.abs(ds - dsc).max() <= 1e-8 * np.abs(dsc).max()


@pytest.mark.parametrize("n", [17, 64, 65, 100, 128])
def test_complex_operators_and_projection(handle, n):
    """Complex K, M and D; Y and H of more than 8 columns."""
    rom, rng = synth.modal_rom(n, 90 + n, 0.02, alpha=1e-4, beta=0.5)
    K, M, D = (a * (1 + 1e-3j) for a in (rom.K, rom.M, rom.D))
    handle.rom_set(0, K, M, D, rom.eta)
    nin, nout = 11, 6
    B, C = synth.complex_normal(rng, (n, nin)), synth.complex_normal(rng, (nout, n))
    handle.rom_set_io(0, B, C)
    freq, load = np.array([4.0, 600.0, 1250.0]), synth.complex_normal(rng, (nin, 2))
    F = np.hstack([B @ load, B])
    Xo, io, _, _ = oracle.sweep(K, M, D, rom.eta, freq, F)
    assert (io == 0).all()
    kappa = synth.cond2(rom, freq).max()
    for mode in ("plain", "refined"):
        X, info, be, _ = handle.sweep(0, freq, F, mode=mode, tol=1e-14)
        assert (info == 0).all() and be.max() <= 1e-14
        assert np.abs(X - Xo).max() <= (2e-14 * kappa * np.sqrt(n) + 1e-14) * np.abs(Xo).max(), mode
        Y, H, info, _ = handle.back_transform(0, freq, load, nin, nout, mode=mode, tol=1e-14)
        assert (info == 0).all()
        R = np.matmul(C, X)
        # the same solutions up to their backward errors, products of n terms: n u
        tol = 2 * (1e-14 + n * 2.2e-16) * kappa * np.sqrt(n)
        assert np.abs(np.concatenate([Y, H], axis=2) - R).max() <= tol * np.abs(R).max(), mode
