"""Times of calls against others of the same handle, where a slower form went unnoticed before:
the best of several runs of each, bounds between what both forms measured."""
import time

import numpy as np
import pytest

from staccato_amd import synth

pytestmark = pytest.mark.gpu


def _best(calls, reps=8):
    """Shortest time of each call, the calls in turn, three at a stretch."""
    import torch
    best = [1e9] * len(calls)
    for f in calls:
        f()
    torch.cuda.synchronize()
    for _ in range(reps):
        for i, f in enumerate(calls):
            t = time.perf_counter()
            for _ in range(3):
                f()
            torch.cuda.synchronize()
            best[i] = min(best[i], time.perf_counter() - t)
    return best


def _buffers(nf, n, nrhs):
    import torch
    return (torch.empty((nf, nrhs, n), dtype=torch.complex128, device="cuda"),
            torch.empty(nf, dtype=torch.int32, device="cuda"),
            torch.empty((nf, nrhs), dtype=torch.float64, device="cuda"))


@pytest.mark.parametrize("n", [144, 176, 256])
def test_explicit_matrices_cost_little_more_than_a_sweep(handle, n):
    """The matrices of a sweep with complex operators, one load, refined: read from HBM
    instead of assembled, 1.00 to 1.08 times the sweep (loads in batches), 1.33 to 1.41
    (one column at a time)."""
    import torch
    nf = 512
    rom, rng = synth.modal_rom(n, n, 0.02)
    freq = np.linspace(1.0, 1200.0, nf)
    A = (1 + 0.02j) * rom.K[None] - ((2 * np.pi * freq) ** 2)[:, None, None] * rom.M[None]
    A_t = torch.from_numpy(np.ascontiguousarray(A.transpose(0, 2, 1))).cuda()
    F_t = torch.from_numpy(synth.complex_normal(rng, (1, n))).cuda()
    B_t, f_t = F_t[None].repeat(nf, 1, 1), torch.from_numpy(freq).cuda()
    X, info, _ = _buffers(nf, n, 1)
    st = torch.cuda.Stream()
    torch.cuda.synchronize()
    handle.rom_set(0, (1 + 0.02j) * rom.K, rom.M, None, 0.0)
    args = dict(mode="refined", tol=1e-12, stream=st.cuda_stream)
    explicit, sweep = _best([lambda: handle.gesv_batched_dev(A_t, B_t, X, info, None, **args),
                             lambda: handle.sweep_dev(0, f_t, F_t, X, info, None, **args)])
    assert (info == 0).all()
    assert explicit <= 1.2 * sweep, explicit / sweep


@pytest.mark.parametrize("n,nrhs", [(100, 1), (112, 2), (128, 1), (128, 4)])
def test_backward_errors_cost_little(handle, n, nrhs):
    """Plain sweep with Rayleigh damping: 1.05 to 1.07 times the sweep without them
    (every wavefront works on them), 1.21 to 1.27 (one wavefront per load)."""
    import torch
    nf = 1024
    rom, rng = synth.modal_rom(n, n, 0.01, alpha=1e-4, beta=0.5)
    handle.rom_set(0, rom.K, rom.M, rom.D, rom.eta)
    f_t = torch.linspace(1.0, 1200.0, nf, dtype=torch.float64, device="cuda")
    F_t = torch.from_numpy(synth.complex_normal(rng, (nrhs, n))).cuda()
    X, info, be = _buffers(nf, n, nrhs)
    st = torch.cuda.Stream()
    torch.cuda.synchronize()
    with_be, without = _best([lambda: handle.sweep_dev(0, f_t, F_t, X, info, be, stream=st.cuda_stream),
                              lambda: handle.sweep_dev(0, f_t, F_t, X, info, None, stream=st.cuda_stream)])
    assert (info == 0).all() and be.max() <= 1e-13
    assert with_be <= 1.15 * without, with_be / without


@pytest.mark.parametrize("n", [24, 37, 64, 70, 71, 72, 128])
@pytest.mark.parametrize("nrhs", [1, 2, 3, 4, 5, 10, 17])
def test_backward_errors_of_every_split(handle, n, nrhs):
    """One wavefront per load or all of them, with U's room large enough for their sums or
    not: the errors that X has."""
    rom, rng = synth.modal_rom(n, 30 + n, 0.02, alpha=1e-4, beta=0.5)
    handle.rom_set(0, rom.K, rom.M, rom.D, rom.eta)
    freq = np.array([3.0, 500.0])
    F = synth.complex_normal(rng, (n, nrhs)) * 10.0 ** rng.uniform(-3, 3, nrhs)
    X, info, be, _ = handle.sweep(0, freq, F, mode="plain")
    assert (info == 0).all()
    for j, f in enumerate(freq):
        A = synth.assemble(rom, f)
        den = np.abs(A).sum(1).max() * np.abs(X[j]).max(0) + np.abs(F).max(0)
        ref = np.abs(F - A @ X[j]).max(0) / den
        # both residuals round by at most (n + 4) u of |A| |x| + |b| a row
        assert np.abs(be[j] - ref).max() <= 2 * (n + 4) * 2.0 ** -52
        assert be[j].max() <= n * 2.0 ** -52 + 1e-15


@pytest.mark.parametrize("ops", ["real", "explicit"])
@pytest.mark.parametrize("rounds", [2, 3, 6])
def test_one_refined_load_takes_the_faster_kernel(handle, rounds, ops):
    """n = 112: where the points fill three workgroups per CU, the register panel is 5 to 12 %
    faster than the register kernel's two, a round of two the other way round by 20 %;
    the automatic choice is never much slower than the panel."""
    import torch
    n, nf = 112, rounds * torch.cuda.get_device_properties(0).multi_processor_count
    rom, rng = synth.modal_rom(n, n, 0.02)
    handle.rom_set(0, rom.K, rom.M, None, rom.eta)
    f_t = torch.linspace(1.0, 1200.0, nf, dtype=torch.float64, device="cuda")
    F_t = torch.from_numpy(synth.complex_normal(rng, (1, n))).cuda()
    X, info, be = _buffers(nf, n, 1)
    st = torch.cuda.Stream()
    args = dict(mode="refined", tol=1e-12, stream=st.cuda_stream)
    if ops == "explicit":
        w2 = (2 * np.pi * f_t.cpu().numpy()) ** 2
        A = (1 + 0.02j) * rom.K[None] - w2[:, None, None] * rom.M[None]
        A_t, B_t = torch.from_numpy(A.transpose(0, 2, 1).copy()).cuda(), F_t[None].repeat(nf, 1, 1)
    torch.cuda.synchronize()

    def run(kernel):
        def call():
            handle.set_policy(n, "refined", kernel)
            if ops == "explicit":
                handle.gesv_batched_dev(A_t, B_t, X, info, be, **args)
            else:
                handle.sweep_dev(0, f_t, F_t, X, info, be, **args)
        return call

    try:
        auto, panel = _best([run(None), run(1)])
    finally:
        handle.clear_policies()
    assert (info == 0).all() and be.max() <= 1e-12
    assert auto <= 1.045 * panel, auto / panel


@pytest.mark.parametrize("n,nrhs,berr", [(128, 16, False), (128, 33, True), (100, 128, True), (112, 64, False), (32, 256, False)])
def test_many_plain_loads_take_the_faster_kernel(handle, n, nrhs, berr):
    """The register kernel factors again for every 16 loads (8 up to n = 64): beyond that the
    kernels that factor once are up to 1.4 times as fast, at 16 loads slower by a third;
    the automatic choice is never much slower than they."""
    import torch
    nf = 2 * torch.cuda.get_device_properties(0).multi_processor_count
    rom, rng = synth.modal_rom(n, n, 0.02)
    handle.rom_set(0, rom.K, rom.M, None, rom.eta)
    f_t = torch.linspace(1.0, 1200.0, nf, dtype=torch.float64, device="cuda")
    F_t = torch.from_numpy(synth.complex_normal(rng, (nrhs, n))).cuda()
    X, info, be = _buffers(nf, n, nrhs)
    st = torch.cuda.Stream()
    torch.cuda.synchronize()

    def run(kernel):
        def call():
            handle.set_policy(n, "plain", kernel)
            handle.sweep_dev(0, f_t, F_t, X, info, be if berr else None, stream=st.cuda_stream)
        return call

    try:
        auto, once = _best([run(None), run(1)], reps=4)
    finally:
        handle.clear_policies()
    assert (info == 0).all()
    assert auto <= 1.045 * once, auto / once
