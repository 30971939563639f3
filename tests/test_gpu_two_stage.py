"""Sizes at the edges of the kernels that a grid's lengths choose, on the GPU against the oracle.

One-dimensional grids: the direct convolution's lane and chunk counts change at 64 and 128 points and it ends
at 256; longer ones take the generic kernels. Two-dimensional grids (one slab) run whole runs of steps in one
launch. Real-space sweeps: lanes per line and the LDS pitch change at multiples of 16 and at 1024 points.

Bars: FP64 1e-10 relative as in the other oracle tests; FP32 2e-5, the stated error of that form.
"""
import numpy as np
import pytest

from oracle import oracle as O
from tests.conftest import golden

pytestmark = pytest.mark.gpu


def say(msg):
    print(msg, flush=True)


def rel(a, b):
    a, b = np.asarray(a), np.asarray(b)
    return float(np.max(np.abs(a - b)) / max(np.max(np.abs(b)), 1e-300))


@pytest.fixture(scope="module")
def capi():
    from langevin_fts_amd import capi as c
    return c


@pytest.fixture(scope="module")
def ctx(capi):
    return capi.Context(0)


def check(ctx, capi, name, model, nx, prec="fp64", mask=None, bc=None, stress=True):
    plan = golden("plans")[f"{name}|{model}|0"]
    inp = plan["input"]
    M = int(np.prod(nx))
    rng = np.random.default_rng(23)
    w = {m: 0.6 * rng.standard_normal(M) for m in inp["bonds"]}
    # Real-space steps: a right side carries a rounding error of about 4 r eps of q, r = b^2 ds / (12 dx^2), which
    # the solve passes on at long wavelengths. At 2.3 over 1023 points (r of 800 or more, some 100 steps) that
    # alone is 1e-10 on Q, oracle included; at dx = 0.05 it is below 1e-12.
    lx = [2.3 + 0.4 * i if bc is None else 0.05 * n for i, n in enumerate(nx)]
    ref = O.Solver(O.Grid(nx, lx, mask), plan, inp["ds"], inp["bonds"], inp["solvents"], realspace_bc=bc)
    ref.compute_statistics(w)
    g = capi.Grid(ctx, nx, lx, mask)
    P = capi.Plan(plan, inp["ds"], inp["bonds"], plan["schedules"]["4"], inp["solvents"])
    s = capi.Solver(g, P, capi.FTS_FP64 if prec == "fp64" else capi.FTS_FP32, realspace_bc=bc)
    bar = 1e-10 if prec == "fp64" else 2e-5
    for again in range(2):
        s.compute_statistics(w)
        for p in range(len(plan["polymers"])):
            assert abs(s.get_total_partition(p) / ref.get_total_partition(p) - 1) < bar
        for m in inp["bonds"]:
            assert rel(s.get_total_concentration(m), ref.get_total_concentration(m)) < bar
    if stress and bc is None:
        s.compute_stress()
        ref.compute_stress()
        assert rel(s.get_stress(), ref.get_stress()) < (bar if prec == "fp64" else 1e-4)


MODELS = [("branched", "continuous"), ("diblock_f0.5_ds1_90", "discrete")]


@pytest.mark.parametrize("name,model", MODELS)
@pytest.mark.parametrize("n", [2, 30, 63, 64, 65, 126, 128, 130, 255, 256])
def test_lines(ctx, capi, n, name, model):
    say(f"line {n} {model}")
    check(ctx, capi, name, model, [n])


@pytest.mark.parametrize("name,model", MODELS)
@pytest.mark.parametrize("nx", [[4, 4], [21, 26], [22, 35], [33, 64], [60, 104]])
def test_flat_grids(ctx, capi, nx, name, model):
    say(f"flat {nx} {model}")
    rng = np.random.default_rng(4)
    check(ctx, capi, name, model, nx)
    check(ctx, capi, name, model, nx, mask=(rng.random(int(np.prod(nx))) > 0.1).astype(np.float64), stress=False)


@pytest.mark.parametrize("nx", [[100], [45, 32], [27, 10, 16], [15, 18, 25]])
def test_fp32(ctx, capi, nx):
    say(f"fp32 {nx}")
    check(ctx, capi, "diblock_f0.5_ds1_90", "discrete", nx, "fp32")


# FP32: a segment's factors are 2^-24 off or so at every point, in every step: 2e-5 is 300 segments' worth where all
# act the same way, so chains of 100 segments keep it (the branched one has 276, with masks Q is 4e-6 and 2.04e-5 off)
MODELS32 = [("diblock_f0.36_ds0.01", "continuous"), ("diblock_f0.5_ds1_90", "discrete")]


@pytest.mark.parametrize("name,model", MODELS32)
@pytest.mark.parametrize("nx", [[2], [64], [72], [128], [135], [256], [20, 48], [60, 64], [100, 150]])
def test_fp32_lines_and_flat_grids(ctx, capi, nx, name, model):
    """FP32 instances of the one-launch kernels, at the lengths where the line kernel's lanes and chunks change."""
    say(f"fp32 one launch {nx} {model}")
    check(ctx, capi, name, model, nx, "fp32")
    rng = np.random.default_rng(4)
    check(ctx, capi, name, model, nx, "fp32", mask=(rng.random(int(np.prod(nx))) > 0.1).astype(np.float64), stress=False)


@pytest.mark.parametrize("nx", [[48] * 3, [64] * 3, [40, 45, 36]])
def test_fp32_keeps_the_mean(ctx, capi, nx):
    """The field's mean is not rounded to an FP32 sum of all points in every convolution: 100 continuous steps round that 300
    times, 1e-6 on Q (measured rms of these fields with the mean in the x transform: 1.1e-6, 1.0e-6, 1.1e-6). Past
    the x transform it keeps the planes' rounding: some 12 additions of 2^-24 / sqrt(12) each way, 6e-8 of a plane's mean,
    over sqrt(nx) planes and sqrt(2 x 300) passes: 1.8e-7 at nx = 64. The bar on the rms of 6 fields is 2.5 times that;
    the value is the FP64 solver's Q."""
    plan = golden("plans")["diblock_f0.36_ds0.01|continuous|0"]
    inp = plan["input"]
    M = int(np.prod(nx))
    g = capi.Grid(ctx, nx, [0.07 * n for n in nx])
    P = capi.Plan(plan, inp["ds"], inp["bonds"], plan["schedules"]["4"])
    s64, s32 = capi.Solver(g, P, capi.FTS_FP64), capi.Solver(g, P, capi.FTS_FP32)
    err = []
    for seed in range(6):
        rng = np.random.default_rng(seed)
        w = {m: 2.0 * rng.standard_normal(M).astype(np.float32).astype(np.float64) for m in inp["bonds"]}
        s64.compute_propagators(w)
        s32.compute_propagators(w)
        err.append(s32.get_total_partition(0) / s64.get_total_partition(0) - 1)
    rms = float(np.sqrt(np.mean(np.square(err))))
    say(f"fp32 mean {nx}: Q errors {' '.join('%+.1e' % e for e in err)}, rms {rms:.1e}")
    assert rms < 2.5 * 1.8e-7 * np.sqrt(64 / nx[0])


@pytest.mark.parametrize("n", [15, 16, 17, 512, 1023, 1024, 1025])
def test_realspace_lines(ctx, capi, n):
    say(f"real-space sweeps {n}")
    check(ctx, capi, "branched", "continuous", [n], bc=["periodic", "periodic"])
    if n < 1000 or n == 1024:
        check(ctx, capi, "branched", "continuous", [n, 3],
              bc=["absorbing", "reflecting", "periodic", "periodic"])


@pytest.mark.parametrize("prec,n", [("fp64", 260), ("fp64", 512), ("fp64", 1001), ("fp64", 2187), ("fp32", 300),
                                    ("fp64", 4096), ("fp64", 4500)])
def test_long_lines(ctx, capi, prec, n):
    """One-dimensional grids beyond the direct convolution: a row of the slab pass must fit its threads."""
    say(f"long line {n} {prec}")
    for name, model in MODELS[1:] if prec == "fp32" else MODELS:
        check(ctx, capi, name, model, [n], prec)


def test_two_long_rows(ctx, capi):
    say("2 x 5000")
    check(ctx, capi, *MODELS[1], [2, 5000])


def test_rows_beyond_the_lds_are_refused(ctx, capi):
    """A line of 5120 points has no slab plan: the pseudo-spectral solver says so, real-space steps take it."""
    plan = golden("plans")["diblock_f0.5_ds1_16|continuous|0"]
    inp = plan["input"]
    g = capi.Grid(ctx, [5120], [6.0])
    P = capi.Plan(plan, inp["ds"], inp["bonds"], plan["schedules"]["4"])
    with pytest.raises(RuntimeError, match="LDS"):
        capi.Solver(g, P)
    capi.Solver(g, P, realspace_bc=["periodic", "periodic"])
