"""Performance cases of the framework: the calls a memetic reconstruction makes.

A case is one call (or a short list of operations) on a population that is
resident on the GPU, at the grid sizes, population sizes, block lengths and
constraint settings of this repository's schedules (workloads.py), settings
(settings.py), tests and benchmark:

  iterate    an ER/HIO/RAAR schedule segment between two shrink-wraps
  sw         one shrink-wrap of the population
  evaluate   the errors and the symmetry of every individual
  align      the alignment of the population to a reference density
  crossover  the children of the population (host densities in and out)
  loss       the differentiable Fourier loss, forward and backward

Populations are late-stage ones: the object (overlapping projected ellipsoids
with a smooth phase) plus a per-individual perturbation of 0.2 % inside a
support a few pixels larger than it, with the detector's beamstop, gaps and
saturated pixels masked. `scale` is the object's size relative to the
repository's 512^2 ellipsoid workload (semi-axes 20 - 60 px of 512), so the
support covers a sixth to nearly all of the rows.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from s_spi_spring_amd import grad, hipcore, spring_core

DEV = "cuda"


def listed():
    return [
        # One block of the 512^2 schedule: population 64, RAAR 25 (the benchmark's step).
        dict(name="raar 512 pop 64", op="iterate", n=512, population=64, scale=1.0, reality=0.0,
             seq="RAAR 25 0.87"),
        # The default settings' generation segment: HIO 40, ER 40, popsize 128, reality 0.5.
        dict(name="hio-er 256 pop 128", op="iterate", n=256, population=128, scale=1.0, reality=0.5,
             seq="HIO 40 0.95;ER 40"),
        # The 128^2 schedule's mixed block with its population of 8: the smallest call.
        dict(name="hio-er 128 pop 8", op="iterate", n=128, population=8, scale=1.0, reality=0.0,
             seq="HIO 10 0.9;ER 10"),
        # A large population of small fields.
        dict(name="hio 128 pop 256", op="iterate", n=128, population=256, scale=1.0, reality=0.0,
             seq="HIO 20 0.9"),
        # The large-pattern block.
        dict(name="raar 1024 pop 32", op="iterate", n=1024, population=32, scale=0.8, reality=0.0,
             seq="RAAR 25 0.87"),
        # A ragged population of a non-power-of-two size with a wide object, and the closing ER block.
        dict(name="raar-er 768 pop 11", op="iterate", n=768, population=11, scale=1.5, reality=0.0,
             seq="RAAR 25 0.87;ER 25"),
        # One individual per call, as a caller of the per-individual interface runs it.
        dict(name="hio 512 pop 1", op="iterate", n=512, population=1, scale=1.0, reality=0.0,
             seq="HIO 25 0.95"),
        # The shrink-wrap after every block.
        dict(name="sw 512 pop 64", op="sw", n=512, population=64, scale=1.0, sigma=2.0, threshold=0.03),
        # The fitness of the population at the end of a sequence.
        dict(name="evaluate 512 pop 64", op="evaluate", n=512, population=64, scale=1.0, reality=0.0),
        # The alignment to the best individual before averaging.
        dict(name="align 384 pop 37", op="align", n=384, population=37, scale=1.0),
        # A generation's children (the default crossover weights).
        dict(name="crossover 512 pop 24", op="crossover", n=512, population=24, scale=1.0),
        # One forward and backward pass of the loss in a PyTorch program.
        dict(name="loss 1024 pop 8", op="loss", n=1024, population=8, scale=0.8, kind="poisson"),
    ]


# Pixels of a drawn population by size: at most those of 32 fields of 1024^2.
_MAX_PIXELS = 32 * 1024 * 1024
_MAX_POP = {64: 512, 128: 512, 256: 256, 384: 128, 512: 96, 768: 40, 1024: 32, 2048: 8}


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    op = rng.choice(["iterate"] * 6 + ["sw", "evaluate", "align", "crossover", "loss", "loss"])
    sizes = [64, 128, 256, 384, 512, 768, 1024, 2048] if op == "iterate" else [256, 384, 512, 768, 1024]
    n = rng.choice(sizes)
    pop = _log_int(rng, 1, min(_MAX_POP[n], _MAX_PIXELS // (n * n)))
    scale = round(math.exp(rng.uniform(math.log(0.5), math.log(1.7))), 3)
    case = dict(op=op, n=n, population=pop, scale=scale)
    if op == "iterate":
        alg = rng.choice(["RAAR", "HIO", "HIO", "RAAR", "ER"])
        budget = min(40, 22 * _MAX_PIXELS // (pop * n * n))       # iterations: no dearer than the listed cases
        it = rng.randint(10, budget)
        seq = f"ER {it}" if alg == "ER" else f"{alg} {it} {round(rng.uniform(0.8, 0.95), 3)}"
        if alg != "ER" and it + 6 <= budget and rng.random() < 0.6:
            seq += f";ER {rng.randint(5, budget - it - 1)}"
        case.update(reality=rng.choice([0.0, 0.0, 0.5]), seq=seq)
    elif op == "sw":
        case.update(sigma=round(rng.uniform(1.5, 3.0), 3), threshold=rng.choice([0.03, 0.2]))
    elif op == "evaluate":
        case.update(reality=rng.choice([0.0, 0.5]))
    elif op == "crossover":
        case.update(population=min(pop, 24))
    elif op == "loss":
        case.update(kind=rng.choice(["poisson", "amplitude"]))
    return case


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------
def _object(n, scale, gen):
    """1-5 overlapping projected ellipsoids: semi-axes 20-60 px and centres within
    80 px of the middle at n = 512 and scale 1, amplitude 0.5-1, phase within
    +-0.5 rad (float64, complex)."""
    u = torch.rand(64, generator=gen, dtype=torch.float64).tolist()
    s = scale * n / 512.0
    y, x = torch.meshgrid(torch.arange(n, dtype=torch.float64, device=DEV),
                          torch.arange(n, dtype=torch.float64, device=DEV), indexing="ij")
    thick = torch.zeros(n, n, dtype=torch.float64, device=DEV)
    phase = torch.zeros_like(thick)
    for i in range(1 + int(u[0] * 5)):
        v = u[1 + 9 * i:10 + 9 * i]
        a, b = (20 + 40 * v[0]) * s, (20 + 40 * v[1]) * s
        rc, tc, th = 80 * s * math.sqrt(v[2]), 2 * math.pi * v[3], math.pi * v[4]
        dx, dy = x - n / 2 - rc * math.cos(tc), y - n / 2 - rc * math.sin(tc)
        xr, yr = dx * math.cos(th) + dy * math.sin(th), -dx * math.sin(th) + dy * math.cos(th)
        q = 1 - (xr / a) ** 2 - (yr / b) ** 2
        thick += q.clamp(min=0).sqrt()
        ramp = ((2 * v[5] - 1) * xr / a + (2 * v[6] - 1) * yr / b + 2 * v[7] - 1) * 0.25
        phase += torch.where(q > 0, ramp, torch.zeros_like(ramp))
    amp = torch.where(thick > 0, 0.5 + 0.5 * thick / thick.max(), torch.zeros_like(thick))
    return torch.polar(amp, phase.clamp(-0.5, 0.5))


def _ft(rho):
    """Unnormalised transform with kernel exp(+2 pi i k.x/N)."""
    return torch.fft.ifft2(rho, norm="forward")


def _ift(f):
    """The inverse of _ft: kernel exp(-2 pi i k.x/N), divided by N^2."""
    return torch.fft.fft2(f, norm="forward")


def _detector_mask(n, gen):
    """Masked pixels, corner origin: a 12 px beamstop and two 4 px gaps (at 512^2)
    and 0.5 % saturated pixels."""
    c = torch.arange(n, device=DEV)
    c = torch.minimum(c, n - c).to(torch.float64)
    m = (c[:, None] ** 2 + c[None, :] ** 2) <= (12 * n / 512) ** 2
    gap = c < 2
    m = m | gap[:, None] | gap[None, :]
    return m | (torch.rand(n, n, generator=gen, dtype=torch.float64) < 0.005).to(DEV)


def _inputs(case, seed):
    """(corner-origin amplitude, densities, supports): complex64 and bool tensors."""
    n, P = case["n"], case["population"]
    gen = torch.Generator().manual_seed(seed)
    obj = _object(n, case["scale"], gen)
    p = _ft(obj).abs() ** 2
    photons = 1e8 if case["op"] == "loss" else 1e9
    lam = p * (photons / p.sum())
    rho = obj * math.sqrt(photons / float(p.sum()))
    if case["op"] == "loss":                   # low counts: the likelihood's noise
        dgen = torch.Generator(device=DEV).manual_seed(seed + 1)
        lam = torch.poisson(lam, generator=dgen)
    amp = torch.where(_detector_mask(n, gen), torch.full_like(lam, -1.0), lam.sqrt()).to(torch.float32)
    # two pixels of margin, but none where the phase constraint tests them: their
    # values are the perturbation alone, whose phase is anything
    grow = 0 if case.get("reality") else 2
    supp = torch.nn.functional.max_pool2d((obj.abs() > 0).to(torch.float32)[None, None], 2 * grow + 1, 1, grow)[0, 0] > 0
    dgen = torch.Generator(device=DEV).manual_seed(seed + 2)
    noise = torch.randn(P, n, n, 2, generator=dgen, device=DEV, dtype=torch.float32)
    pert = torch.view_as_complex(noise) * (0.002 * float(rho.abs().max())) * supp
    dens = rho.to(torch.complex64)[None] + pert
    return amp, dens, supp


class _DeviceArray:
    """The array interface of a field batch that `owner` holds on the device."""

    def __init__(self, ptr, shape, typestr, owner):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": shape, "typestr": typestr, "data": (ptr, False), "version": 3}


def _view(ptr, shape, typestr, owner):
    """Tensor over the owner's memory; the tensor keeps the owner, and so the memory, alive."""
    t = torch.as_tensor(_DeviceArray(ptr, shape, typestr, owner), device=DEV)
    t.owner = owner
    return t


class _State:
    pass


def prepare(case, seed):
    n, P = case["n"], case["population"]
    amp, dens, supp = _inputs(case, seed)
    st = _State()
    st.case = case
    if case["op"] == "align":                   # copies of the object moved about the grid
        gen = torch.Generator().manual_seed(seed + 3)
        st.moves = torch.randint(0, n, (P, 2), generator=gen).tolist()
        ref = dens[0].cpu().numpy()
        dens = torch.stack([torch.roll(d, m, (0, 1)) for d, m in zip(dens, st.moves)])
        st.ref, st.phase = ref, np.full(P, 0.25, np.float32)
    if case["op"] == "crossover":
        counts = torch.where(amp >= 0, amp * amp, amp)
        pr = spring_core.phase_retrieval
        st.solver = pr.Solver(torch.fft.fftshift(counts).cpu().numpy(), reality=0.0, nthreads=8, use_bounds=False,
                              gpus=[0], seed=seed % 1000 + 1)
        s32 = supp.cpu().numpy().astype(np.int32)
        st.recs = [pr.Reconstruction(d, s32) for d in dens.cpu().numpy()]
        st.solver.Evaluate(st.recs)
        st.best = min(st.recs, key=lambda r: r.get_error())
        st.avg = st.solver.GetAverage(st.recs, fraction=0.8)
        return st
    st.be = hipcore.Backend(amp.cpu().numpy(), capacity=P)
    if case["op"] == "loss":
        st.rho = dens.clone().requires_grad_(True)
        return st
    st.be.set_population(dens.cpu().numpy(), np.broadcast_to(supp.cpu().numpy(), (P, n, n)))
    if case["op"] == "iterate":
        st.seq = []
        for o in case["seq"].split(";"):
            w = o.split()
            st.seq.append((w[0], [float(v) for v in w[1:]]))
    rho, s8, _ = st.be.device_buffers()
    st.rho = _view(rho, (P, n, n, 2), "<f4", st.be)
    st.supp = _view(s8, (P, n, n), "|u1", st.be)
    return st


def run(st):
    c = st.case
    if c["op"] == "iterate":
        st.be.run(st.seq, 1, c["reality"])
        return st.rho
    if c["op"] == "sw":
        st.be.sw(c["sigma"], c["threshold"])
        return st.supp
    if c["op"] == "evaluate":
        return st.be.evaluate(c["reality"])
    if c["op"] == "align":
        return {"shifts": st.be.align(st.ref, st.phase, st.phase), "rho": st.rho}
    if c["op"] == "crossover":
        children = st.solver.Crossover(st.recs, st.best, st.avg, 0.6, 0.4, 1.0, 1.0, False, 0.0)
        return [[r.get_density(), r.get_support()] for r in children]
    st.rho.grad = None
    loss = grad.fourier_loss(st.rho, st.be, c["kind"])
    loss.sum().backward()
    return {"loss": loss.detach(), "grad": st.rho.grad}


# ---------------------------------------------------------------------------
# Minimal work of one pass
# ---------------------------------------------------------------------------
def work(case):
    """Bytes: the state read once and written once (densities 8 B/px, supports 1
    B/px, the amplitude once). Flops: 5 N^2 log2(N^2) per 2-D transform that the
    operation is made of, and the pixel arithmetic is not counted."""
    n, P = case["n"], case["population"]
    px, fft = float(n * n * P), 10.0 * n * n * math.log2(n) * P
    amp = 4.0 * n * n
    if case["op"] == "iterate":
        its = sum(int(o.split()[1]) + 1 for o in case["seq"].split(";"))
        return {"bytes": 17 * px + amp, "flops": 2 * its * fft}
    if case["op"] == "sw":
        return {"bytes": 9 * px + amp, "flops": 4 * fft}
    if case["op"] == "evaluate":
        return {"bytes": 9 * px + amp, "flops": 5 * fft}
    if case["op"] == "align":
        return {"bytes": 18 * px + amp + 8.0 * n * n, "flops": 3 * fft}
    if case["op"] == "crossover":
        return {"bytes": 18 * px + 2 * amp + 8.0 * n * n, "flops": 12 * fft}
    return {"bytes": 16 * px + amp, "flops": 2 * fft}


# ---------------------------------------------------------------------------
# The same results in double precision
# ---------------------------------------------------------------------------
def _project(F, amp):
    m = F.abs()
    return torch.where((amp >= 0) & (m > 0), F * (amp / m.clamp(min=1e-300)), F)


def _accept(z, supp, reality):
    """Support pixels whose phase lies within +-pi (1 - reality)."""
    return supp & (z.angle().abs() < math.pi * (1 - reality))


def _iterate64(case, amp, rho, supp):
    for o in case["seq"].split(";"):
        w = o.split()
        beta = float(np.float32(float(w[2]))) if len(w) > 2 else 0.0
        for _ in range(int(w[1])):
            d = _ift(_project(_ft(rho), amp))
            if w[0] == "ER":
                rho = torch.where(_accept(d, supp, case["reality"]), d, torch.zeros_like(d))
            elif w[0] == "HIO":
                rho = torch.where(_accept(d, supp, case["reality"]), d, rho - beta * d)
            else:
                ok = _accept(2 * d - rho, supp, case["reality"])
                rho = torch.where(ok, d, beta * rho + (1 - 2 * beta) * d)
        rho = _ift(_project(_ft(rho), amp))
    return rho


def _errors64(amp, rho, supp, reality):
    ok = _accept(rho, supp, reality)
    rs = torch.where(ok, rho, torch.zeros_like(rho))
    F = _ft(rs)
    m = F.abs()
    k = (amp >= 0).expand_as(m)
    z = torch.zeros_like(m)
    ef = (torch.where(k, (amp - m) ** 2, z).sum((1, 2)) / torch.where(k, (amp ** 2).expand_as(m), z).sum((1, 2))).sqrt()
    d = _ift(_project(F, amp))
    out = ~supp
    er = (torch.where(out, d.imag ** 2, z).sum((1, 2)) / (d.abs() ** 2).sum((1, 2))).sqrt()
    return {"error_fourier": ef, "error_real": er, "complexsum": m.amax((1, 2)), "modulesum": rs.abs().sum((1, 2))}


def exact(case, seed):
    if case["op"] in ("sw", "crossover"):
        return None
    amp, dens, supp = _inputs(case, seed)
    a64 = amp.to(torch.float64)
    n, P = case["n"], case["population"]
    if case["op"] == "align":
        turn = complex(math.cos(float(np.float32(0.25))), math.sin(float(np.float32(0.25))))
        return {"shifts": None, "rho": torch.view_as_real(dens.to(torch.complex128) * turn)}
    if case["op"] == "loss":
        x = dens.to(torch.complex128).requires_grad_(True)
        u = _ft(x).abs() ** 2
        if case["kind"] == "poisson":
            term = u - a64 * a64 * torch.log(u + float(np.float32(1e-3)))
        else:
            term = (u.sqrt() - a64) ** 2
        loss = torch.where(a64 >= 0, term, torch.zeros_like(term)).sum((1, 2))
        loss.sum().backward()
        return {"loss": loss.detach(), "grad": x.grad}
    parts = []
    step = max(1, (1 << 23) // (n * n))
    for i in range(0, P, step):
        r = dens[i:i + step].to(torch.complex128)
        if case["op"] == "iterate":
            parts.append(torch.view_as_real(_iterate64(case, a64, r, supp)))
        else:
            parts.append(_errors64(a64, r, supp, case["reality"]))
    if case["op"] == "evaluate":
        got = {k: torch.cat([q[k] for q in parts]).cpu().numpy() for k in parts[0]}
        got["symmetry"] = None
        return got
    return torch.cat(parts)
