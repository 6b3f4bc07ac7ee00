"""GPU: beam and field state entry points: beam info, per-slice current
(which scales the deposited source linearly), and the device field copy
(planes and ring state, bit for bit)."""
from __future__ import annotations

import time

import numpy as np
import pytest

import cases
from cases import LAMBDA0, quad_step
from genesis4_cuda_port_amd import api

pytestmark = pytest.mark.gpu

from test_gpu_parity import gpu_beam, gpu_field, noisy_field, relerr  # noqa: E402


@pytest.mark.parametrize("prec", [api.FP64, api.MIXED])
def test_beam_info(gpu_ctx, prec):
    c = cases.make_case(nslice=5, npart=128, ngrid=17)
    b = gpu_beam(gpu_ctx, c, prec)
    assert b.info() == (5, 5 * 128, prec)
    b.close()


def test_current_scales_the_source(gpu_ctx):
    """From a zero field, one field step is the source term alone, linear in
    the slice current: doubling the current of two slices doubles their
    planes and leaves the others as they were."""
    c = cases.make_case(nslice=4, npart=2048, ngrid=33)
    st = quad_step()
    z = np.zeros(c.nslice * c.ngrid ** 2)

    def step(current):
        b = gpu_beam(gpu_ctx, c)
        b.set_current(current)
        f = gpu_field(gpu_ctx, c, re=z, im=z)
        f.track(b, st, st.delz)
        re, im, _ = f.download()
        f.close()
        b.close()
        return (re + 1j * im).reshape(c.nslice, -1)

    cur = np.array(c.beam.current, dtype=float)
    a = step(cur)
    scale = np.array([1.0, 2.0, 1.0, 2.0])
    b = step(cur * scale)
    assert np.abs(a).max() > 0
    for s in range(c.nslice):
        assert relerr(b[s], scale[s] * a[s]) < 1e-13


@pytest.mark.parametrize("prec", [api.FP64, api.MIXED])
def test_field_copy_is_exact(gpu_ctx, prec):
    c = cases.make_case(nslice=6, npart=64, ngrid=21, seed_power=1e5)
    re, im = noisy_field(c, scale=0.5)
    src = gpu_field(gpu_ctx, c, prec, re=re, im=im, first=3)
    src.set_ring(3, 0.25)
    dst = gpu_field(gpu_ctx, c, prec)
    dst.copy_from(src)
    a, b = src.download(), dst.download()
    assert np.array_equal(a[0], b[0]) and np.array_equal(a[1], b[1]) and a[2] == b[2] == 3
    assert dst.ring() == (3, 0.25)
    src.close()
    dst.close()


@pytest.mark.parametrize("prec", [api.FP64, api.MIXED])
def test_new_field_is_cleared_before_its_planes_are_set(prec):
    """A field's planes are zeroed on its context's stream, so planes set next
    stay: each new field, filled at once by a kernel on that stream, holds the
    plane everywhere."""
    print(f"case field_create_order prec={prec}", flush=True)
    rng = np.random.default_rng(5)
    n, g = 64, 129
    re, im = rng.standard_normal(g * g), rng.standard_normal(g * g)
    want = (re + 1j * im) if prec == api.FP64 else (re + 1j * im).astype(np.complex64)
    with api.Context(0) as ctx:
        for _ in range(4):
            f = api.Field(ctx, prec, n, g, 0.3e-3, LAMBDA0, LAMBDA0)
            f.fill_planes(re, im)
            fr, fi, _ = f.download()
            assert np.array_equal((fr + 1j * fi).reshape(n, -1), np.broadcast_to(want, (n, g * g)))
            f.close()


def test_fp64_passes_queue_without_the_host_waiting():
    """60 FP64 passes queued behind about 20 ms of work: each uploads its
    parameter block through a ring of 64 slots, so none of them waits for the
    device and the host is done with them long before it."""
    print("case queue_depth", flush=True)
    c = cases.make_case(nslice=256, npart=2048, ngrid=101, nsteps=200,
                        seed_power=1e4)
    small = cases.make_case(nslice=4, npart=256, ngrid=17)
    st = quad_step()
    with api.Context(0) as ctx:
        work, f = gpu_beam(ctx, c, api.MIXED), gpu_field(ctx, c, api.MIXED)
        b = gpu_beam(ctx, small, api.FP64)
        shares = []
        for _ in range(3):
            run = api.Run(ctx, work, f, c.steps, LAMBDA0, c.sample, True, False, 1, False)
            b.track_transverse(st, 1e-3, False)  # the ring's memory, on the first call
            ctx.synchronize()
            run.advance(len(c.steps))
            t0 = time.perf_counter()
            for k in range(60):
                b.track_transverse(st, 1e-3, bool(k % 2))
            t1 = time.perf_counter()
            ctx.synchronize()
            t2 = time.perf_counter()
            shares.append((t1 - t0) / (t2 - t0))
            run.close()
        print(f"  host share of the queue's time {shares}", flush=True)
        for x in (b, work, f):
            x.close()
    assert min(shares) < 0.5
