"""Performance cases: the work a user of the solver has it do, through its
public entry points, from the smallest grid to the largest that is measured.

Four kinds of case:
  run       the `dns` program's loop: RK4 steps with the energy / enstrophy
            line every 10 steps, then the spectral state read out (as for a
            checkpoint) into page-locked host memory;
  dump      the same loop with `-d`: pressure kept, and after every 10 steps a
            snapshot of U, V, W, P through the asynchronous snapshot calls;
  ensemble  a batch of simulations of mixed grid sizes and viscosities, ten
            steps per call, then every member's state read out;
  gradient  the discrete adjoint: final enstrophy and its gradient with
            respect to the initial velocity, with checkpoints, device to
            device as the torch binding calls it.

A pass continues from the state that the last one left, as a program's time
loop does (the gradient starts from its initial field each time).

Grids go up to 648^3: three states of a 1024^3 grid do not fit the card
(FP64 takes 160 GB), and each case keeps a page-locked buffer of its state.
"""
import ctypes
import math

import numpy as np
import torch
from torch.utils.checkpoint import checkpoint

import dns_amd

# viscosities of the Taylor-Green sweep: 1/Re
REYNOLDS = (100, 200, 400, 800, 1600, 3000)
# every grid size the library carries up to the largest measured
SIZES = (8, 12, 16, 18, 24, 32, 36, 48, 54, 64, 72, 96, 108, 128, 144, 162, 192, 216, 256, 288, 324, 384, 432, 486,
         512, 576, 648)


def listed():
    return [
        # smallest calls: launches and latency are everything
        {"name": "run-16", "kind": "run", "n": 16, "precision": "fp64", "re": 100, "steps": 10},
        # the README's Taylor-Green sample (n=64), a student's laptop run
        {"name": "run-64", "kind": "run", "n": 64, "precision": "fp64", "re": 100, "steps": 50},
        # the reference's Reynolds sweep at its coarse and its fine grid
        {"name": "run-128", "kind": "run", "n": 128, "precision": "fp64", "re": 1600, "steps": 20},
        {"name": "run-256", "kind": "run", "n": 256, "precision": "fp64", "re": 1600, "steps": 10},
        # a grid of threes in mixed precision: pencils that fill no wavefront
        {"name": "run-162-mixed", "kind": "run", "n": 162, "precision": "mixed", "re": 800, "steps": 20},
        # the mixed form with double accumulation, radix-3 grid
        {"name": "run-384-acc64", "kind": "run", "n": 384, "precision": "mixed_acc64", "re": 3000, "steps": 10},
        # the headline workload in both precisions
        {"name": "run-512", "kind": "run", "n": 512, "precision": "fp64", "re": 3000, "steps": 10},
        {"name": "run-512-mixed", "kind": "run", "n": 512, "precision": "mixed", "re": 3000, "steps": 20},
        # the largest grid, beyond the sizes that carry several launch shapes
        {"name": "run-648-mixed", "kind": "run", "n": 648, "precision": "mixed", "re": 3000, "steps": 10},
        # `dns -d`: a snapshot every 10 steps
        {"name": "dump-216", "kind": "dump", "n": 216, "precision": "fp64", "re": 1600, "steps": 20},
        # the 24-member ensemble: 4 grids x 6 Reynolds numbers
        {"name": "ensemble-24", "kind": "ensemble", "sizes": "64 96 128 192", "per_size": 6, "precision": "mixed",
         "steps": 20},
        # the adjoint workload's grid, with a checkpoint interval per ten steps
        {"name": "gradient-128", "kind": "gradient", "n": 128, "re": 800, "steps": 20, "every": 10},
    ]


def draw(rng):
    kind = rng.choice(("run", "run", "run", "run", "dump", "ensemble", "gradient"))
    re = rng.choice(REYNOLDS)

    def size(lo, hi):
        at = math.exp(rng.uniform(math.log(lo), math.log(hi)))
        return min(SIZES, key=lambda n: abs(math.log(n / at)))

    if kind == "run":
        n = size(8, 648)
        # a pass stays below the cost of the largest listed one
        precision = rng.choice(("fp64", "mixed", "mixed_acc64") if n <= 512 else ("mixed",))
        return {"kind": kind, "n": n, "precision": precision, "re": re,
                "steps": rng.choice((10, 20, 30, 40, 50)) if n <= 256 else 10}
    if kind == "dump":
        return {"kind": kind, "n": size(16, 288), "precision": rng.choice(("fp64", "mixed")), "re": re,
                "steps": rng.choice((10, 20, 30))}
    if kind == "ensemble":
        sizes = sorted({size(16, 192) for _ in range(rng.randint(2, 5))})
        return {"kind": kind, "sizes": " ".join(map(str, sizes)), "per_size": rng.randint(1, 6),
                "precision": rng.choice(("fp64", "mixed", "mixed_acc64")), "steps": rng.choice((10, 20))}
    return {"kind": kind, "n": size(16, 144), "re": re, "steps": rng.randint(4, 20), "every": rng.randint(2, 10)}


def _time_step(n):
    # advective number k_max max|u| dt well below the RK4 bound (2.8); the
    # headline workload's 5e-4 at n=512
    return 0.256 / n


def _velocity(n, seed):
    """Taylor-Green plus a seeded random velocity whose spectrum fills the
    whole grid (k^-5/3 beyond the energy-carrying scales), [3][n][n][n]
    doubles on the GPU."""
    gen = torch.Generator(device="cuda").manual_seed(int(seed) % (1 << 31) + 77777 * n)
    x = torch.arange(n, device="cuda", dtype=torch.float64) * (2 * math.pi / n)
    s, c = x.sin(), x.cos()
    u = torch.zeros((3, n, n, n), device="cuda", dtype=torch.float64)
    u[0] = s[:, None, None] * c[None, :, None] * c[None, None, :]
    u[1] = -c[:, None, None] * s[None, :, None] * c[None, None, :]
    m = torch.fft.fftfreq(n, 1.0 / n, device="cuda", dtype=torch.float64)
    k2 = (m * m)[:, None, None] + (m * m)[None, :, None] + (m * m)[None, None, : n // 2 + 1]
    amp = (1.0 + k2 / 9.0).pow_(-11.0 / 12.0)
    del k2
    for f in range(3):
        w = torch.fft.rfftn(torch.randn((n, n, n), device="cuda", dtype=torch.float64, generator=gen))
        w *= amp
        r = torch.fft.irfftn(w, s=(n, n, n))
        del w
        u[f] += 0.3 * r / r.std()
        del r
    return u


def _load(n, seed, call, out):
    """call(numpy velocity) with a page-locked copy of the initial field,
    which the state buffer `out` has room for."""
    host = torch.view_as_real(out).reshape(-1)[: 3 * n ** 3].view(3, n, n, n)
    host.copy_(_velocity(n, seed))
    call(host.numpy())


def _state_buffer(n):
    return torch.empty((3, n, n, n // 2 + 1), dtype=torch.complex128, pin_memory=True)


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("run", "dump"):
        n = case["n"]
        s = dns_amd.Solver(n, 1.0 / case["re"], _time_step(n), case["precision"])
        out = _state_buffer(n)
        _load(n, seed, s.load_velocity, out)
        if kind == "run":
            return {"case": case, "solver": s, "out": out}
        s.set_pressure_capture(True)
        return {"case": case, "solver": s}
    if kind == "ensemble":
        ns, nus = _members(case)
        b = dns_amd.Batch(ns, nus, [_time_step(n) for n in ns], case["precision"])
        out = [_state_buffer(n) for n in ns]
        for m, n in enumerate(ns):
            _load(n, seed + 1000 * m, lambda u, m=m: b.load_velocity(m, u), out[m])
        return {"case": case, "batch": b, "out": out}
    n = case["n"]
    return {"case": case, "solver": dns_amd.Solver(n, 1.0 / case["re"], _time_step(n)), "u0": _velocity(n, seed),
            "grad": torch.empty((3, n, n, n), device="cuda", dtype=torch.float64)}


def _members(case):
    sizes = [int(n) for n in case["sizes"].split()]
    ns = [n for n in sizes for _ in range(case["per_size"])]
    return ns, [1.0 / REYNOLDS[m % len(REYNOLDS)] for m in range(len(ns))]


def _check(rc):
    if rc != dns_amd.DNS_OK:
        raise dns_amd.DnsError(rc, "perf case")


class _Snapshot:
    """Keeps a solver alive for as long as its page-locked snapshot is used."""

    def __init__(self, solver, address, n):
        self.solver = solver
        self.__array_interface__ = {"shape": (4, n, n, n), "typestr": "<f8", "data": (address, False), "version": 3}


def run(state):
    case, lib = state["case"], dns_amd.lib()
    if case["kind"] == "run":
        s, lines = state["solver"], []
        for _ in range(case["steps"] // 10):
            s.step(10)
            lines.append(s.diagnostics())
        _check(lib.dns_get_spectral(s._ctx, ctypes.c_void_p(state["out"].data_ptr())))
        return {"lines": torch.tensor(lines, dtype=torch.float64), "state": state["out"]}
    if case["kind"] == "dump":
        s, lines = state["solver"], []
        # the snapshot of one ten-step segment is copied while the next runs
        for _ in range(case["steps"] // 10):
            s.step(10)
            lines.append(s.diagnostics())
            s.snapshot_begin()
        p = ctypes.POINTER(ctypes.c_double)()
        _check(lib.dns_snapshot_wait(s._ctx, ctypes.byref(p)))
        address = ctypes.cast(p, ctypes.c_void_p).value
        return {"lines": torch.tensor(lines, dtype=torch.float64), "snapshot": np.asarray(_Snapshot(s, address, case["n"]))}
    if case["kind"] == "ensemble":
        b, lines = state["batch"], []
        for _ in range(case["steps"] // 10):
            b.step(10)
            lines.append([b.diagnostics(m) for m in range(len(b))])
        for m, out in enumerate(state["out"]):
            _check(lib.dns_batch_get_spectral(b._b, m, ctypes.c_void_p(out.data_ptr())))
        return {"lines": torch.tensor(lines, dtype=torch.float64), "states": state["out"]}
    s, z = state["solver"], ctypes.c_double()
    torch.cuda.synchronize()  # the library works on its own stream
    _check(lib.dns_adjoint_forward(s._ctx, ctypes.c_void_p(state["u0"].data_ptr()), case["steps"], case["every"],
                                   ctypes.byref(z)))
    _check(lib.dns_adjoint_backward(s._ctx, 1.0, ctypes.c_void_p(state["grad"].data_ptr())))
    return {"enstrophy": torch.tensor(z.value, dtype=torch.float64), "grad": state["grad"]}


def work(case):
    """A step reads the state (three spectral fields in double and the
    physical velocity of the last stage) and writes it; 33 real transforms
    of 2.5 N log2 N operations and about 150 more per point.  A gradient runs
    every step forward twice and backward once (about twice the transforms).
    Results are written once more where they are read out."""
    def step(n, precision):
        spectral, points = 16.0 * n * n * (n // 2 + 1), float(n) ** 3
        real = 8 if precision == "fp64" else 4
        return 2 * (3 * spectral + 3 * real * points), 33 * 2.5 * points * math.log2(points) + 150 * points, 3 * spectral

    if case["kind"] == "ensemble":
        b = f = 0.0
        for n in _members(case)[0]:
            sb, sf, out = step(n, case["precision"])
            b += case["steps"] * sb + out
            f += case["steps"] * sf
        return {"bytes": b, "flops": f}
    sb, sf, out = step(case["n"], case.get("precision", "fp64"))
    if case["kind"] == "gradient":
        return {"bytes": 4 * case["steps"] * sb, "flops": 4 * case["steps"] * sf}
    if case["kind"] == "dump":
        out *= 8.0 / 3.0 * case["steps"] // 10
    return {"bytes": case["steps"] * sb + out, "flops": case["steps"] * sf}


def tolerance(case):
    """Four times the largest error against exact() over the listed cases and
    24 drawn ones: 2.2e-15 (gradient) and 1e-12 of the root mean square in
    FP64, 1.1e-7 and 6.5e-5 in the mixed forms."""
    if case.get("precision", "fp64") == "fp64":
        return {"rel": 1e-14, "max": 4e-12}
    return {"rel": 4e-7, "max": 3e-4}


# ---------------------------------------------------------------------------
# The same in plain torch, in 64 bits.
A = (1 / 6.0, 1 / 3.0, 1 / 3.0, 1 / 6.0)
B = (0.5, 0.5, 1.0, 0.0)


class _Spectral:
    """Wavenumbers, dealias mask and transforms of one grid."""

    def __init__(self, n):
        self.n = n
        i = torch.arange(n, device="cuda")
        m = torch.where(i < n // 2, i, i - n).double()
        k = torch.arange(n // 2 + 1, device="cuda").double()
        self.k = (m[:, None, None], m[None, :, None], k[None, None, :])
        kmax = 2.0 / 3.0 * (n // 2 + 1)
        self.mask = ((self.k[0].abs() < kmax) & (self.k[1].abs() < kmax) & (self.k[2].abs() < kmax)).double()
        self.kk = self.k[0] ** 2 + self.k[1] ** 2 + self.k[2] ** 2

    def fwd(self, f):
        return torch.fft.fftn(torch.fft.rfft(f, dim=2), dim=(0, 1))

    def inv(self, f):
        # unnormalised sums over x and y, then c2r over z, which takes the
        # real parts only at kz = 0 and kz = n/2; 1/n^3 in all
        g = torch.fft.ifftn(f, dim=(0, 1))
        ends = torch.zeros_like(g)
        ends[..., 0], ends[..., -1] = g[..., 0].imag, g[..., -1].imag
        return torch.fft.irfft(g - 1j * ends, n=self.n, dim=2)

    def diagnostics(self, U):
        e = sum(u.real ** 2 + u.imag ** 2 for u in U)
        s = 1.0 / float(self.n) ** 6
        return e.sum() * s, (self.kk * e).sum() * s

    def step(self, U, stale, nu, dt):
        """One RK4 step: the first stage's velocity is the last stage's of
        the step before.  Returns the state, the new stale velocity and the
        last stage's pressure."""
        kx, ky, kz = self.k
        Ur, acc, u, P = U, U, stale, None
        for r in range(4):
            if r:
                u = [self.inv(f) for f in Ur]
            w = [self.inv(1j * f) for f in (ky * Ur[2] - kz * Ur[1], kz * Ur[0] - kx * Ur[2], kx * Ur[1] - ky * Ur[0])]
            N = (u[1] * w[2] - u[2] * w[1], u[2] * w[0] - u[0] * w[2], u[0] * w[1] - u[1] * w[0])
            del w
            d = [self.fwd(f) * (self.mask * dt) for f in N]
            del N
            P = (d[0] * kx + d[1] * ky + d[2] * kz) / self.kk.clamp(min=1.0)
            d = [d[f] - P * self.k[f] - (nu * dt) * self.kk * Ur[f] for f in range(3)]
            acc = [acc[f] + A[r] * d[f] for f in range(3)]
            if r < 3:
                Ur = [U[f] + B[r] * d[f] for f in range(3)]
            del d
        return acc, u, P


def _exact_run(n, nu, dt, u0, steps):
    g = _Spectral(n)
    U, u, P, lines = [g.fwd(f) for f in u0], list(u0), None, []
    for i in range(steps):
        U, u, P = g.step(U, u, nu, dt)
        if i % 10 == 9:
            lines.append([v.item() for v in g.diagnostics(U)])
    return g, U, P, torch.tensor(lines, dtype=torch.float64)


def exact(case, seed):
    kind = case["kind"]
    if kind in ("run", "dump"):
        n = case["n"]
        if float(n) ** 3 * case["steps"] > 5e9:  # over 20 seconds
            return None
        g, U, P, lines = _exact_run(n, 1.0 / case["re"], _time_step(n), _velocity(n, seed), case["steps"])
        if kind == "run":
            return {"lines": lines, "state": torch.stack(U)}
        return {"lines": lines, "snapshot": torch.stack([g.inv(f) for f in (*U, P)])}
    if kind == "ensemble":
        ns, nus = _members(case)
        lines, states = [], []
        for m, n in enumerate(ns):
            _, U, _, got = _exact_run(n, nus[m], _time_step(n), _velocity(n, seed + 1000 * m), case["steps"])
            lines.append(got)
            states.append(torch.stack(U).cpu())
        return {"lines": torch.stack(lines, dim=1), "states": states}
    n = case["n"]
    g, u0 = _Spectral(n), _velocity(n, seed).requires_grad_(True)
    U, u = [g.fwd(f) for f in u0], list(u0)
    for _ in range(case["steps"]):  # a step's inner fields are computed again for its gradient
        U, u = checkpoint(lambda *a: g.step(a[:3], a[3:], 1.0 / case["re"], _time_step(n))[:2], *U, *u,
                          use_reentrant=False)
    z = g.diagnostics(U)[1]
    z.backward()
    return {"enstrophy": z.detach(), "grad": u0.grad}
