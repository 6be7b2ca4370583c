"""FP64 iterations whose undecided pixels can be taken either way.

An update accepts a pixel or not by whether a phase is pi. Where the FP64 value is
nearer to the negative real axis than four times the FP32 oracle's error, either
decision is right, and an iteration that took the other one ends up to 1e-3 apart
(at 768^2, ER, one pixel of test_gpu_wide_supports' 615 rows does: the same in the
form that stores the state). A result beyond a bar has to meet it after up to three
such decisions are taken the other way.
"""
import numpy as np
import scipy.fft

from conftest import rel_l2


def ft(x):
    return scipy.fft.ifft2(x, norm="forward", workers=8)


def ift(x):
    return scipy.fft.fft2(x, norm="forward", workers=8)


def iterate64(orc, alg, beta, rho, supp, amp, flips=(), near=None):
    """Two FP64 iterations and the trailing projection, with the decisions (iteration,
    flat pixel) of `flips` taken the other way; `near` collects the undecided ones."""
    b, a64 = rho.astype(np.complex128), amp.astype(np.float64)
    for it in range(2):
        d = ift(orc.project(ft(b), a64))
        z = 2 * d - b if alg == "RAAR" else d
        accept = (supp != 0) & ~((z.real < 0) & (z.imag == 0))
        if near is not None:
            err = np.abs(orc.ift(orc.project(orc.ft(b.astype(np.complex64)), amp)) - d).max()
            close = (supp != 0) & (z.real < 0) & (np.abs(z.imag) <= (12 if alg == "RAAR" else 4) * err)
            near += [(abs(z.imag.flat[i]), it, i) for i in np.flatnonzero(close)]
        for at, i in flips:
            if at == it:
                accept.flat[i] = not accept.flat[i]
        b = np.where(accept, d, {"ER": 0 * d, "HIO": b - beta * d, "RAAR": beta * b + (1 - 2 * beta) * d}[alg])
    return ift(orc.project(ft(b), a64))


def nearest_decisions(orc, alg, beta, rho, supp, amp, got, bar):
    """Relative L2 to the FP64 iteration after up to three undecided pixels, the least
    decided ones first, and these."""
    near, flips = [], []
    e = rel_l2(got, iterate64(orc, alg, beta, rho, supp, amp, near=near))
    near = [f[1:] for f in sorted(near)]
    while e >= bar and len(flips) < 3:
        best = None
        for f in near:
            if f in flips:
                continue
            ef = rel_l2(got, iterate64(orc, alg, beta, rho, supp, amp, flips + [f]))
            if ef < e:
                e, best = ef, f
            if e < bar:
                break
        if best is None:
            break
        flips.append(best)
    return e, flips
