"""Results of host-memory calls: pieces of the pinned staging memory (8 MiB), rows that a
piece splits, and a leading dimension beyond n, against the same sweep on device memory."""
import ctypes

import numpy as np
import pytest

from staccato_amd import sweep as sw
from staccato_amd import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,nfreq,nrhs,pad", [(33, 1, 1, 0), (33, 7, 2, 3), (57, 5301, 2, 0), (57, 5301, 2, 5),
                                              (31, 16913, 1, 0)])
def test_pieces_and_leading_dimension(handle, n, nfreq, nrhs, pad):
    import torch
    rom, rng = synth.modal_rom(n, 60 + n, 0.02)
    F = synth.complex_normal(rng, (n, nrhs))
    freq = np.linspace(2.0, 1500.0, nfreq)
    handle.rom_set(0, rom.K, rom.M, rom.D, rom.eta)
    dev = torch.device("cuda", 0)
    X_t = torch.empty((nfreq, nrhs, n), dtype=torch.complex128, device=dev)
    info_t = torch.full((nfreq,), 7, dtype=torch.int32, device=dev)
    be_t = torch.empty((nfreq, nrhs), dtype=torch.float64, device=dev)
    handle.sweep_dev(0, torch.from_numpy(freq).to(dev), torch.from_numpy(np.ascontiguousarray(F.T)).to(dev),
                     X_t, info_t, be_t, mode="plain", tol=1e-12)
    torch.cuda.synchronize()
    ldx = n + pad
    Ff = np.asfortranarray(F)
    X = np.full((nfreq, nrhs, ldx), -3.0 + 0j)
    info = np.full(nfreq, 7, dtype=np.int32)
    be = np.empty((nfreq, nrhs))
    st = sw.Stats()
    rc = handle.lib.stc_sweep(handle.h, 0, nfreq, sw._ptr(freq), nrhs, sw._ptr(Ff), n, sw._ptr(X), ldx, sw._ptr(info),
                              sw._ptr(be), sw._mode("plain"), 1e-12, 0, ctypes.byref(st))
    assert rc == 0
    # the same kernels on the same inputs: equal bytes, and nothing written beyond row n
    np.testing.assert_array_equal(X[:, :, :n], X_t.cpu().numpy())
    assert (X[:, :, n:] == -3.0).all()
    np.testing.assert_array_equal(info, info_t.cpu().numpy())
    np.testing.assert_array_equal(be, be_t.cpu().numpy())
    assert st.points == nfreq


def test_back_transform_in_pieces(handle):
    """Y and H interleave per frequency in the buffer (9.6 MB of them here)."""
    n, nin, nout, nfreq, nrhs = 24, 6, 15, 5003, 2
    rom, rng = synth.modal_rom(n, 71, 0.02)
    B, C = synth.complex_normal(rng, (n, nin)), synth.complex_normal(rng, (nout, n))
    load = synth.complex_normal(rng, (nin, nrhs))
    freq = np.linspace(2.0, 1500.0, nfreq)
    handle.rom_set(0, rom.K, rom.M, rom.D, rom.eta)
    handle.rom_set_io(0, B, C)
    Y, H, info, _ = handle.back_transform(0, freq, load, nin, nout, mode="plain", tol=1e-12)
    assert (info == 0).all()
    X, _, _, _ = handle.sweep(0, freq, np.hstack([B @ load, B]), mode="plain", tol=1e-12)
    R = np.matmul(C, X)
    kappa = synth.cond2(rom, freq).max()
    # both solve to a backward error near n u; products of n terms: n u
    tol = 4 * n * 2.2e-16 * kappa * np.sqrt(n)
    assert np.abs(Y - R[:, :, :nrhs]).max() <= tol * np.abs(R).max()
    assert np.abs(H - R[:, :, nrhs:]).max() <= tol * np.abs(R).max()
