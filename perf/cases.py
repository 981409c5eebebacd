"""The measured work of the frequency-sweep library, through its public Python entry points.

A case is one call that a user's program makes on reduced models it has loaded: a
sweep on device tensors or on host arrays, a captured plan over many models, the
adjoint, the back-transformation with transfer functions, a batch of explicit
matrices.  Sizes are those of the repository's workloads (staccato_amd/synth.py),
plus small, odd and ragged ones around them.

Refined sweeps ask for a backward error of 1e-15: the solution then carries the
accuracy of the plain complex128 path, which is what a program that replaces an
FP64 solver by the refined one compares it with.
"""
import math
from concurrent.futures import ThreadPoolExecutor

import numpy as np
import torch

from staccato_amd import Handle, Plan
from staccato_amd._lib import SysDesc

TOL = 1e-15          # refined mode: backward error of FP64 accuracy
SIZES = (32, 48, 64, 96, 128, 192, 256, 384, 512)  # orders met in an uneven batch


def listed():
    return [
        # one user dragging a slider: a handful of frequencies of a very small model
        {"name": "tiny_plain", "kind": "dev", "n": 24, "nfreq": 32, "nrhs": 1, "mode": "plain", "ops": "undamped"},
        # the reference's own call: host arrays, one unit-force load, n = 60
        {"name": "host60_plain", "kind": "host", "n": 60, "nfreq": 1000, "nrhs": 1, "mode": "plain", "ops": "undamped"},
        # a small model of odd order inside an optimisation loop, refined
        {"name": "small47_refined", "kind": "dev", "n": 47, "nfreq": 1501, "nrhs": 2, "mode": "refined", "ops": "rayleigh"},
        # the reference's operators: complex K that already carries (1 + i eta)
        {"name": "complex96_plain", "kind": "dev", "n": 96, "nfreq": 1500, "nrhs": 3, "mode": "plain", "ops": "complex"},
        # an ordinary model of ragged order, refined
        {"name": "mid123_refined", "kind": "dev", "n": 123, "nfreq": 2048, "nrhs": 4, "mode": "refined", "ops": "rayleigh"},
        # gradient of a response objective in every modal stiffness and the loss factor
        {"name": "adjoint128", "kind": "adjoint", "n": 128, "nfreq": 2048, "nrhs": 1, "mode": "plain", "ops": "undamped"},
        # interface Jacobians of coupled models: explicit matrices, one per frequency
        {"name": "gesv64", "kind": "gesv", "n": 64, "nfreq": 4096, "nrhs": 1, "mode": "plain", "ops": "explicit"},
        # responses and transfer functions at a model's inputs and outputs, host arrays
        {"name": "backtransform192", "kind": "back", "n": 192, "nfreq": 800, "nrhs": 1, "nin": 6, "nout": 12,
         "mode": "refined", "ops": "undamped"},
        # the uniform batch, plain and refined
        {"name": "uniform256_plain", "kind": "dev", "n": 256, "nfreq": 4096, "nrhs": 4, "mode": "plain", "ops": "rayleigh"},
        {"name": "uniform256_refined", "kind": "dev", "n": 256, "nfreq": 4096, "nrhs": 4, "mode": "refined",
         "ops": "rayleigh"},
        # many models of different order in one captured launch
        {"name": "uneven_plan", "kind": "plan", "n": 512, "nfreq": 1024, "nrhs": 8, "nsys": 24, "mode": "refined",
         "ops": "undamped"},
        # the largest model, many loads
        {"name": "dense1024_refined", "kind": "dev", "n": 1024, "nfreq": 512, "nrhs": 16, "mode": "refined",
         "ops": "rayleigh"},
    ]


def draw(rng):
    """One more case of the ranges above."""
    def log(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.49)))))

    kind = rng.choice(["dev"] * 6 + ["host", "plan", "adjoint", "gesv", "back"])
    mode = rng.choice(["plain", "refined"])
    ops = rng.choice(["undamped", "rayleigh", "rayleigh", "complex"])
    c = {"kind": kind, "n": log(12, 1024), "nfreq": log(16, 4096), "nrhs": log(1, 16), "mode": mode, "ops": ops}
    if kind == "host":
        c.update(n=log(12, 256), nfreq=log(16, 2048), nrhs=log(1, 4))
    elif kind == "plan":
        c.update(n=rng.choice(SIZES[3:]), nfreq=log(64, 1024), nrhs=log(1, 8), nsys=log(2, 24), mode="refined", ops="undamped")
    elif kind == "adjoint":
        c.update(n=log(16, 256), nfreq=log(64, 2048), nrhs=log(1, 3), mode="plain", ops="undamped")
    elif kind == "gesv":
        c.update(n=log(12, 200), nfreq=log(16, 4096), nrhs=log(1, 4), mode="plain", ops="explicit")
    elif kind == "back":
        c.update(n=log(16, 320), nfreq=log(16, 1500), nrhs=1, nin=log(1, 12), nout=log(1, 200), ops="undamped")
    # no more work than the listed cases: fewer frequencies for the large models
    most = 4e10 if mode == "plain" and c["n"] > 512 else 2e11
    per = work(dict(c, nfreq=1))["flops"]
    c["nfreq"] = max(1, min(c["nfreq"], int(most / per)))
    return c


# ---- inputs ----------------------------------------------------------------------------------------
def _cnormal(rng, *shape):
    return rng.standard_normal(shape) + 1j * rng.standard_normal(shape)


def _rom(n, ops, rng):
    """A model with modes at 10..1000 Hz: K, M, D (or None), eta, Phi, kdiag."""
    Q, R = np.linalg.qr(rng.standard_normal((n, n)))
    Q = Q * np.where(np.diag(R) < 0, -1.0, 1.0)
    m = rng.uniform(0.5, 2.0, n)
    kd = m * (2 * np.pi * 10.0 ** rng.uniform(1.0, 3.0, n)) ** 2

    def form(d):
        A = (Q * d) @ Q.T
        return 0.5 * (A + A.T)

    K, M = form(kd), form(m)
    if ops == "rayleigh":
        return K, M, form(1e-4 * kd + 0.5 * m), 0.01, Q, kd
    if ops == "complex":
        return K * (1 + 0.02j), M, None, 0.0, Q, kd
    return K, M, None, 0.02, Q, kd


def _systems(case, rng):
    """(n, nfreq, nrhs) of every model of a plan."""
    sizes = [s for s in SIZES if s <= case["n"]]
    out = []
    for i in range(case["nsys"]):
        n = case["n"] if i == 0 else int(rng.choice(sizes))
        out.append((n, max(1, int(case["nfreq"] * rng.uniform(0.125, 1.0))), int(rng.integers(1, case["nrhs"] + 1))))
    return out


def _inputs(case, seed):
    rng = np.random.default_rng([seed, case["n"], case["nfreq"]])
    n, nf, nrhs = case["n"], case["nfreq"], case["nrhs"]
    if case["kind"] == "plan":
        # the orders, counts and loads of the batch are the case's, the models the seed's
        shape = np.random.default_rng([7, case["n"], case["nfreq"], case["nsys"]])
        d = []
        for sn, sf, sr in _systems(case, shape):
            d.append({"rom": _rom(sn, case["ops"], rng), "freq": np.linspace(1.0, 1500.0, sf), "F": _cnormal(rng, sn, sr)})
        return d
    d = {"freq": np.linspace(1.0, 1200.0 if n < 200 else 2000.0, nf) + rng.uniform(0.0, 0.2)}
    if case["kind"] == "gesv":
        # compliance-like diagonal over couplings, as an interface Jacobian has
        d["gen"] = int(rng.integers(1 << 40))
        return d
    d["rom"] = _rom(n, case["ops"], rng)
    if case["kind"] == "host":
        d["F"] = np.zeros((n, nrhs), dtype=np.complex128)
        d["F"][rng.choice(n, nrhs, replace=False), np.arange(nrhs)] = 1.0  # unit forces
    elif case["kind"] == "back":
        d["B"], d["C"] = _cnormal(rng, n, case["nin"]), _cnormal(rng, case["nout"], n)
        d["load"] = _cnormal(rng, case["nin"], nrhs)
    else:
        d["F"] = _cnormal(rng, n, nrhs)
    if case["kind"] == "adjoint":
        d["c"] = _cnormal(rng, n)
    return d


def _explicit(case, d):
    """Matrices (batch, n, n) stored column-major and right-hand sides (batch, nrhs, n), on the device."""
    g = torch.Generator(device="cuda").manual_seed(d["gen"])
    n, nb, nrhs = case["n"], case["nfreq"], case["nrhs"]
    A = torch.view_as_complex(torch.randn((nb, n, n, 2), generator=g, device="cuda", dtype=torch.float64))
    A.diagonal(dim1=1, dim2=2).add_(2.0 * math.sqrt(n))
    B = torch.view_as_complex(torch.randn((nb, nrhs, n, 2), generator=g, device="cuda", dtype=torch.float64))
    return A, B


class _State:
    """What the program keeps: a handle with its models, a stream, inputs and output buffers."""

    def __init__(self, case):
        self.case, self.plan, self.h = case, None, Handle(0)
        self.stream = torch.cuda.Stream()

    def __del__(self):
        if self.plan is not None:
            torch.cuda.synchronize()
            self.plan.close()
        self.h.close()


def _dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def prepare(case, seed):
    s = _State(case)
    d = _inputs(case, seed)
    kind, n, nf, nrhs = case["kind"], case["n"], case["nfreq"], case["nrhs"]
    if kind == "plan":
        descs, s.keep, s.out = (SysDesc * len(d))(), [], []
        for i, sy in enumerate(d):
            K, M, D, eta, _, _ = sy["rom"]
            s.h.rom_set(i, K, M, D, eta)
            sn, sr = sy["F"].shape
            sf = sy["freq"].size
            fr, F = _dev(sy["freq"]), _dev(sy["F"].T)
            X = torch.zeros((sf, sr, sn), dtype=torch.complex128, device="cuda")
            info = torch.zeros(sf, dtype=torch.int32, device="cuda")
            s.keep += [fr, F]
            s.out += [X, info]
            e = descs[i]
            e.rom_id, e.nfreq, e.freq_hz, e.nrhs = i, sf, fr.data_ptr(), sr
            e.F, e.ldf, e.X, e.ldx, e.info, e.berr = F.data_ptr(), sn, X.data_ptr(), sn, info.data_ptr(), None
        torch.cuda.synchronize()
        s.plan = Plan(s.h, descs, mode=case["mode"], tol=TOL)
        return s
    s.d = d
    if kind == "gesv":
        s.A, s.B = _explicit(case, d)
    else:
        K, M, D, eta, _, _ = d["rom"]
        s.h.rom_set(0, K, M, D, eta)
    if kind == "back":
        s.h.rom_set_io(0, d["B"], d["C"])
    if kind == "dev":
        s.freq, s.F = _dev(d["freq"]), _dev(d["F"].T)
    if kind in ("dev", "gesv"):
        s.X = torch.zeros((nf, nrhs, n), dtype=torch.complex128, device="cuda")
        s.info = torch.zeros(nf, dtype=torch.int32, device="cuda")
    torch.cuda.synchronize()
    return s


def run(s):
    c, kind, mode = s.case, s.case["kind"], s.case["mode"]
    if kind == "dev":
        s.h.sweep_dev(0, s.freq, s.F, s.X, s.info, mode=mode, tol=TOL, stream=s.stream.cuda_stream)
        return s.X, s.info
    if kind == "plan":
        s.plan.execute(s.stream.cuda_stream)
        return s.out
    if kind == "gesv":
        s.h.gesv_batched_dev(s.A, s.B, s.X, s.info, mode=mode, tol=TOL, stream=s.stream.cuda_stream)
        return s.X, s.info
    d = s.d
    if kind == "host":
        X, info, _, _ = s.h.sweep(0, d["freq"], d["F"], mode=mode, tol=TOL, berr=False)
        return X, info
    if kind == "back":
        Y, H, info, _ = s.h.back_transform(0, d["freq"], d["load"], c["nin"], c["nout"], mode=mode, tol=TOL)
        return Y, H, info
    _, _, _, _, Phi, kd = d["rom"]
    J, ds, de, info = s.h.adjoint(0, d["freq"], d["F"], d["c"], Phi, kd, mode=mode, tol=TOL)
    return J, ds, de, info


def work(case):
    n, nf, nrhs = case["n"], case["nfreq"], case["nrhs"]
    if case["kind"] == "plan":
        b = f = 0.0
        for sn, sf, sr in _systems(case, np.random.default_rng([7, case["n"], case["nfreq"], case["nsys"]])):
            w = work({"kind": "dev", "n": sn, "nfreq": sf, "nrhs": sr, "ops": case["ops"]})
            b, f = b + w["bytes"], f + w["flops"]
        return {"bytes": b, "flops": f}
    ops = {"undamped": 2 * 8, "rayleigh": 3 * 8, "complex": 2 * 16, "explicit": 16 * nf}[case["ops"]] * n * n
    lu = 8.0 / 3.0 * n ** 3
    if case["kind"] == "adjoint":  # two solves, mu^H K x and the p = n modal products
        return {"bytes": ops + 8 * n * n + 16 * n * (nrhs + 1) + 8 * n + 4 * nf,
                "flops": nf * (lu + nrhs * (2 * 8 + 4 + 8) * n * n)}
    if case["kind"] == "back":
        ncol, nin, nout = nrhs + case["nin"], case["nin"], case["nout"]
        return {"bytes": ops + 16 * n * (nin + nout) + nf * (16 * nout * ncol + 4),
                "flops": nf * (lu + ncol * (8.0 * n * n + 8.0 * n * nout))}
    rhs = 16 * n * nrhs * (nf if case["kind"] == "gesv" else 1)
    return {"bytes": ops + rhs + nf * (16 * n * nrhs + 12), "flops": nf * (lu + 8.0 * n * n * nrhs)}


# ---- the same in 64 bits, by LAPACK on the host ------------------------------------------------------
def _each(f, count):
    """[f(0), f(1), ...], one LAPACK thread per item."""
    threads = torch.get_num_threads()
    torch.set_num_threads(1)
    try:
        with ThreadPoolExecutor(16) as pool:
            return list(pool.map(f, range(count)))
    finally:
        torch.set_num_threads(threads)


def _solutions(rom, freq, F, after=lambda A, X: X):
    """after(A, A^-1 F) at every frequency."""
    K, M, D, eta, _, _ = rom
    K, M, F = torch.from_numpy((1 + 1j * eta) * K), torch.from_numpy(M), torch.from_numpy(F)
    D = None if D is None else torch.from_numpy(1j * D)

    def one(j):
        w = 2 * np.pi * float(freq[j])
        A = K - w * w * M
        if D is not None:
            A += w * D
        return after(A, torch.linalg.solve(A, F))

    return _each(one, freq.size)


def exact(case, seed):
    d = _inputs(case, seed)
    kind = case["kind"]
    if kind == "plan":
        out = []
        for sy in d:
            out += [torch.stack(_solutions(sy["rom"], sy["freq"], sy["F"])).transpose(1, 2), None]
        return out
    if kind == "gesv":
        A, B = (t.cpu() for t in _explicit(case, d))
        return torch.stack(_each(lambda j: torch.linalg.solve(A[j].T, B[j].T), case["nfreq"])).transpose(1, 2), None
    freq, rom = d["freq"], d["rom"]
    if kind == "dev":
        return torch.stack(_solutions(rom, freq, d["F"])).transpose(1, 2), None
    if kind == "host":
        return torch.stack(_solutions(rom, freq, d["F"])), None
    if kind == "back":
        C = torch.from_numpy(d["C"])
        Y = torch.stack(_solutions(rom, freq, np.concatenate([d["B"] @ d["load"], d["B"]], 1), lambda A, X: C @ X))
        return Y[:, :, :case["nrhs"]], Y[:, :, case["nrhs"]:], None
    K, _, _, eta, Phi, kd = rom
    c, kd = torch.from_numpy(d["c"]), torch.from_numpy((1 + 1j * eta) * kd)
    K, P = (torch.from_numpy(a).to(torch.complex128) for a in (K, Phi))

    def gradient(A, X):
        g = c.conj() @ X
        mu = torch.linalg.solve(A.mH, torch.outer(c, g))
        ds = -2 * (kd[:, None] * (P.T @ mu).conj() * (P.T @ X)).real.sum(1)
        return float(g.abs().square().sum()), ds, float(2 * (mu.conj() * (K @ X)).sum().imag)

    J, ds, de = zip(*_solutions(rom, freq, d["F"], gradient))
    return math.fsum(J), torch.stack(ds).sum(0), math.fsum(de), None
