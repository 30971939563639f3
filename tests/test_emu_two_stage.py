"""The two-stage FFT kernels of fts_fft_two.hpp, built for the host from their own source by
tests/emu/fft_two_emu.cpp and run as emulated workgroups with AddressSanitizer on the LDS block
and on every global buffer (NaN in what was never written): forward and inverse transforms
against numpy, a convolution with the bond factors, and two masked propagator steps of each kind
by the slab and pencil passes and by the one-launch kernels of flat grids, against numpy in FP64.
The grids take every radix 1..16 as r1 or r2 of each axis, odd and even lengths (rows without a
partner, no Nyquist column), more butterflies than threads, the longest axis and planes that fill the
LDS. CPU only.

Tolerances: a transform's rounding error grows as eps log2(M) in the 2-norm; 64 eps bounds each
result's largest error over its largest value for the steps' 12 transforms at these sizes."""
import fractions
import os
import shutil
import subprocess

import numpy as np
import pytest

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
EMU = os.path.join(REPO, "tests", "emu")
HIP = os.path.join(REPO, "langevin_fts_amd", "csrc", "hip")

pytestmark = pytest.mark.skipif(shutil.which("g++") is None or not os.path.isdir(EMU),
                                reason="needs g++ and tests/emu")


@pytest.fixture(scope="module")
def exe(tmp_path_factory):
    path = str(tmp_path_factory.mktemp("emu") / "fft_two_emu")
    subprocess.run(["g++", "-std=c++17", "-O1", "-fsanitize=address", "-fno-omit-frame-pointer", "-I", EMU,
                    "-I", HIP, "-o", path, os.path.join(EMU, "fft_two_emu.cpp")], check=True, capture_output=True)
    return path


def run(exe, op, esize, n, a, tmp):
    fi, fo = os.path.join(tmp, "in.bin"), os.path.join(tmp, "out.bin")
    dt = np.float32 if esize == 4 else np.float64
    np.ascontiguousarray(a, dtype=dt).tofile(fi)
    r = subprocess.run([exe, op, str(esize)] + [str(x) for x in n] + [fi, fo], capture_output=True, text=True,
                       timeout=600, env=dict(os.environ, ASAN_OPTIONS="detect_leaks=0"))
    assert r.returncode == 0, r.stdout + r.stderr
    return np.fromfile(fo, dtype=dt).astype(np.float64)


def bond(n, share):
    f = 1.0
    for d, L in enumerate(n):
        k = np.arange(L // 2 + 1 if d == 2 else L)
        k = np.minimum(k, L - k)
        f = f * np.exp(-0.3 * share * (k / L) ** 2).reshape([-1 if i == d else 1 for i in range(3)])
    return f


def conv(n, q, share):
    return np.fft.irfftn(bond(n, share) * np.fft.rfftn(q), s=n, axes=(0, 1, 2))


def off(x, y):
    return float(np.max(np.abs(x - y.ravel())) / np.max(np.abs(y)))


def check(exe, n, esize, ops, tmp):
    rng = np.random.default_rng(sum(n))
    q, w = 1.0 + 0.3 * rng.standard_normal(n), rng.standard_normal(n)
    mask = (rng.random(n) > 0.2).astype(np.float64)
    if esize == 4:
        q, w = q.astype(np.float32).astype(np.float64), w.astype(np.float32).astype(np.float64)
    tol = 64 * (2.0 ** -53 if esize == 8 else 2.0 ** -24)
    ds = 0.25
    for op in ops:
        if op == "fft":
            ref = np.fft.rfftn(q)
            got = run(exe, op, esize, n, q, tmp)
            e = off(got, np.stack([ref.real, ref.imag], -1))
        elif op == "ifft":
            ref = np.fft.rfftn(q)
            e = off(run(exe, op, esize, n, np.stack([ref.real, ref.imag], -1), tmp), q)
        elif op == "conv":
            e = off(run(exe, op, esize, n, q, tmp), conv(n, q, 1.0))
        else:
            out, x = [], q
            for _ in range(2):
                if op in ("flatd", "lined"):
                    x = np.exp(-w * ds) * conv(n, x, 1.0) * mask
                else:
                    e2, e4 = np.exp(-w * ds / 2), np.exp(-w * ds / 4)
                    q1 = e2 * conv(n, e2 * x, 1.0)
                    q2 = e4 * conv(n, e2 * conv(n, e4 * x, 0.5), 0.5)
                    x = (4 * q2 - q1) / 3 * mask
                out.append(x)
            got = run(exe, op, esize, n, np.concatenate([q.ravel(), w.ravel(), mask.ravel()]), tmp)
            e = off(got, np.stack(out))
        print(n, esize, op, f"{e:.1e}", flush=True)
        assert e < tol, (n, esize, op, e)


def flat_ops(n):
    return (["flat", "flatd"] if n[0] == 1 else []) + (["line", "lined"] if n[0] == n[1] == 1 else [])


# (x, y, z): odd and even lengths of every radix; test_grids_take_every_radix
GRIDS = [(2, 8, 8), (3, 6, 10), (4, 12, 9), (5, 15, 16), (7, 14, 26), (11, 22, 33), (13, 21, 35), (2, 45, 20),
         (6, 7, 13), (1, 60, 104), (1, 1, 128), (1, 1, 30), (2, 30, 27), (9, 10, 1), (16, 3, 4), (2, 49, 25),
         (1, 9, 11), (3, 1, 24), (208, 3, 2), (225, 2, 2), (196, 1, 3), (144, 2, 5), (2, 169, 6), (1, 225, 8),
         (1, 240, 4), (2, 182, 5), (1, 256, 6), (1, 144, 10), (1, 6, 196), (1, 4, 225), (1, 3, 240), (1, 2, 256),
         (1, 5, 144), (1, 2, 182), (60, 1, 2), (72, 1, 2)]
# planes of 140 KB and more of LDS
PLANES = [(1, 126, 126), (1, 84, 182), (1, 112, 128)]
GRIDS32 = [(2, 8, 8), (3, 6, 10), (5, 15, 16), (1, 20, 48), (1, 1, 128), (225, 2, 2), (240, 2, 2), (144, 1, 3),
           (100, 2, 3), (72, 1, 2), (1, 225, 4), (1, 256, 3), (2, 150, 5), (1, 144, 4), (1, 72, 8), (1, 3, 225),
           (1, 2, 256), (1, 4, 144), (1, 2, 64), (1, 100, 150), (1, 1, 72), (1, 1, 256), (1, 3, 9), (24, 1, 2),
           (1, 36, 2)]
LINES = [(1, 1, 2), (1, 1, 63), (1, 1, 64), (1, 1, 65), (1, 1, 130), (1, 1, 225), (1, 1, 256)]


def two_axis(L, y, fp32):
    """fts_two_plan.hpp's rule: the smallest larger radix; on y the first radix is even, or the larger one of an odd
    length; FP32 has no 7, 11 or 13"""
    ok = [r for r in range(1, 17) if not (fp32 and any(r % p == 0 for p in (7, 11, 13)))]
    m, s = next((m, s) for m in ok for s in ok if s <= m and m * s == L)
    return (m, s) if y and (L % 2 == 1 or s % 2 == 1) else (s, m)


def test_grids_take_every_radix():
    for axis in range(3):
        for fp32, grids in ((False, GRIDS + PLANES + LINES), (True, GRIDS32)):
            seen = {r for n in grids for r in two_axis(n[axis], axis == 1, fp32)}
            assert seen >= {r for r in range(1, 17) if not fp32 or r % 7 and r % 11 and r % 13}, (axis, fp32, seen)


@pytest.mark.parametrize("n", LINES)
def test_lines_fp64(exe, n, tmp_path):
    check(exe, n, 8, ["line", "lined"], str(tmp_path))


@pytest.mark.parametrize("n", PLANES)
def test_full_planes_fp64(exe, n, tmp_path):
    check(exe, n, 8, ["conv", "flat"], str(tmp_path))


@pytest.mark.parametrize("n", GRIDS)
def test_two_stage_fp64(exe, n, tmp_path):
    ops = ["fft", "ifft", "conv", "step"] + flat_ops(n)
    check(exe, n, 8, ops, str(tmp_path))


@pytest.mark.parametrize("n", GRIDS32)
def test_two_stage_fp32(exe, n, tmp_path):
    ops = ["fft", "ifft", "conv", "step"] + flat_ops(n)
    check(exe, n, 4, ops, str(tmp_path))


@pytest.mark.parametrize("n", [1, 2, 3, 16, 30, 64, 105, 128, 256])
def test_line_coefficients(exe, n, tmp_path):
    """The coefficients of a line's direct convolutions act the same way in every step: each within an ulp or two of
    the bond factors' inverse transform (longdouble), and their sum, which scales the field's mean, 1 to 2^-60 (the
    rounding of the largest one alone would leave 2^-54, 1e-14 of the mean after 100 steps)."""
    c = run(exe, "linec", 8, (1, 1, n), np.ones(3 * n), str(tmp_path)).reshape(2, n)
    k = np.arange(n // 2 + 1)
    for row, share in zip(c, (0.3, 0.15)):
        b = np.exp(-share * k * k / n / n)
        ref = np.fft.irfft(b.astype(np.longdouble), n) if n > 1 else b.astype(np.longdouble)
        assert ref.dtype == np.longdouble
        exact = sum((fractions.Fraction(float(x)) for x in row), fractions.Fraction(-1))
        print(n, share, f"sum - 1 {float(exact):.1e}", f"coefficients {float(np.max(np.abs(row - ref))):.1e}")
        assert abs(exact) < 2.0 ** -60
        assert np.max(np.abs(row - ref)) < 2 * 2.0 ** -53


@pytest.mark.parametrize("esize,bars", [(8, (0.53, 0.88)), (4, (1.92, 0.53))])
def test_step_factors(exe, esize, bars, tmp_path):
    """The factors exp(-w ds/2) and exp(-w ds/4) of a continuous step against longdouble. FP64: a rounded value (0.5 ulp,
    and the exponential's own 0.02) and its rounded root (half of that relative error, at most sqrt(2) / 4 ulp of the
    root, and 0.5 more). FP32: a product of two rounded values (twice the error, at most sqrt(2) ulp of the product,
    and 0.5 more) and a rounded value."""
    n = (1, 1, 256)
    w = np.random.default_rng(8).uniform(-40, 40, 256)
    if esize == 4:
        w = w.astype(np.float32).astype(np.float64)
    got = run(exe, "factor", esize, n, np.concatenate([w, w, w]), str(tmp_path)).reshape(2, -1)
    for row, coef, bar in zip(got, (0.125, 0.0625), bars):
        ref = np.exp(-w.astype(np.longdouble) * coef)
        ulp = np.spacing(ref.astype(np.float32 if esize == 4 else np.float64)).astype(np.longdouble)
        e = float(np.max(np.abs(row - ref) / ulp))
        print(esize, coef, f"{e:.2f} ulp")
        assert e < bar


def test_step_factors_at_their_limits(exe, tmp_path):
    """Factors of walls and wells: 0, infinity and NaN pass, tiny and huge ones keep their precision (FP64)."""
    w = np.array([np.inf, -np.inf, np.nan, 4000.0, -4000.0, 1e300, -1e300, 0.0])
    got = run(exe, "factor", 8, (1, 1, 8), np.concatenate([w, w, w]), str(tmp_path)).reshape(2, -1)
    for row, coef in zip(got, (0.125, 0.0625)):
        with np.errstate(over="ignore"):
            ref = np.exp(-w * coef)
        assert np.allclose(row, ref, rtol=1e-13, atol=0.0, equal_nan=True), (row, ref)
