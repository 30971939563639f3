"""fts_grid_fft_backward_noalloc (no reference counterpart: the allocation-free form of
fts_grid_fft_backward for callers that cannot allocate) against fts_grid_fft_backward,
called through the C ABI: bit-identical results on two calls in a row on one GPU, the
second with a smaller input, and a clear error for a grid beyond its workspace."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def say(msg):
    print(msg, flush=True)


def spectra(g, capi, batch, dt, seed):
    """batch forward transforms of random real fields, as the backward input"""
    a = np.random.default_rng(seed).standard_normal((batch, g.M)).astype(dt)
    x = capi.DeviceArray.from_host(a)
    spec = capi.DeviceArray(batch * g.Mc * 2 * np.dtype(dt).itemsize)
    g.fft_forward(x.ptr, spec.ptr, batch, capi.FTS_FP64 if dt == np.float64 else capi.FTS_FP32)
    return a, spec


def backward_both(ctx, capi, g, spec, batch, dt):
    p = capi.FTS_FP64 if dt == np.float64 else capi.FTS_FP32
    out_ref = capi.DeviceArray(batch * g.M * np.dtype(dt).itemsize)
    out_na = capi.DeviceArray(batch * g.M * np.dtype(dt).itemsize)
    g.fft_backward(spec.ptr, out_ref.ptr, batch, p)
    capi.check(capi.lib().fts_grid_fft_backward_noalloc(g.h, p, ctypes.c_void_p(spec.ptr),
                                                        ctypes.c_void_p(out_na.ptr), batch))
    ctx.synchronize()
    return out_ref.download((batch, g.M), dt), out_na.download((batch, g.M), dt)


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
def test_noalloc_backward_equals_backward(prec):
    from langevin_fts_amd import capi

    dt = np.float64 if prec == "fp64" else np.float32
    ctx = capi.Context(0)
    # first call: 128^3 batch 3 (one spectrum per chunk of the workspace in FP64),
    # second call: a smaller grid and batch, on the same device workspace
    for shape, batch in [((128, 128, 128), 3), ((48, 40, 36), 2)]:
        say(f"noalloc backward {prec} {shape} batch {batch}")
        g = capi.Grid(ctx, list(shape), [1.0] * 3)
        a, spec = spectra(g, capi, batch, dt, seed=sum(shape) + batch)
        ref, na = backward_both(ctx, capi, g, spec, batch, dt)
        assert np.array_equal(ref, na)
        tol = 1e-12 if prec == "fp64" else 3e-6
        assert np.max(np.abs(na - a)) < tol * np.max(np.abs(a))


def test_noalloc_backward_refuses_grid_beyond_workspace():
    from langevin_fts_amd import capi

    ctx = capi.Context(0)
    say("noalloc backward: 512x128x64 FP64 (34.6 MB of spectrum) exceeds the workspace")
    g = capi.Grid(ctx, [512, 128, 64], [1.0] * 3)
    spec = capi.DeviceArray(g.Mc * 16)
    out = capi.DeviceArray(g.M * 8)
    rc = capi.lib().fts_grid_fft_backward_noalloc(g.h, capi.FTS_FP64, ctypes.c_void_p(spec.ptr),
                                                  ctypes.c_void_p(out.ptr), 1)
    assert rc != 0
    assert b"workspace" in capi.lib().fts_last_error()


@pytest.mark.parametrize("shape", [(256, 180, 64), (240, 96, 160), (256, 63, 256)])
def test_noalloc_backward_takes_grids_up_to_its_workspace(shape):
    """Grids whose half spectrum fits the 32 MiB, in contiguous rows, are taken: 24.3, 29.9 and 33.3 MB."""
    from langevin_fts_amd import capi

    ctx = capi.Context(0)
    say(f"noalloc backward {shape}")
    g = capi.Grid(ctx, list(shape), [1.0] * 3)
    assert g.Mc * 16 <= 32 << 20
    a, spec = spectra(g, capi, 1, np.float64, seed=7)
    ref, na = backward_both(ctx, capi, g, spec, 1, np.float64)
    assert np.array_equal(ref, na)
    assert np.max(np.abs(na - a)) < 1e-12 * np.max(np.abs(a))


@pytest.mark.parametrize("shape,prec", [((48, 40, 36), "fp64"), ((48, 40, 36), "fp32"), ((1, 60, 104), "fp64"),
                                        ((1, 60, 100), "fp32"), ((9, 10, 15), "fp64"), ((9, 10, 15), "fp32"),
                                        ((17, 6, 10), "fp64")])
def test_transforms_of_general_grids(shape, prec):
    """Grids without N^3 kernels transform the caller's contiguous rows: batches beyond one launch, every value of
    every spectrum, with a guard behind the last row, against numpy (eps log2 M is 2e-15 and 1e-6)."""
    from langevin_fts_amd import capi

    dt = np.float64 if prec == "fp64" else np.float32
    p = capi.FTS_FP64 if prec == "fp64" else capi.FTS_FP32
    ctx = capi.Context(0)
    say(f"transforms {shape} {prec}")
    batch, guard = 35, 64
    g = capi.Grid(ctx, list(shape), [1.0] * 3)
    a = np.random.default_rng(sum(shape)).standard_normal((batch,) + shape).astype(dt)
    x = capi.DeviceArray.from_host(a)
    spec = capi.DeviceArray.from_host(np.full(batch * g.Mc * 2 + guard, 7.0, dt))
    g.fft_forward(x.ptr, spec.ptr, batch, p)
    raw = spec.download((batch * g.Mc * 2 + guard,), dt).astype(np.float64)
    assert np.all(raw[-guard:] == 7.0)
    out = raw[:-guard].reshape(batch, g.Mc, 2)
    ref = np.fft.rfftn(a.astype(np.float64), axes=(1, 2, 3)).reshape(batch, -1)
    bar = 1e-14 if prec == "fp64" else 3e-6
    assert np.max(np.abs(out[..., 0] + 1j * out[..., 1] - ref)) < bar * np.max(np.abs(ref))
    g.fft_backward(spec.ptr, x.ptr, batch, p)
    back = x.download(a.shape, dt)
    assert np.max(np.abs(back - a)) < bar * np.max(np.abs(a))
