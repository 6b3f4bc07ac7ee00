"""GPU: segmented ADI sweeps at the edges of their segment lengths.

Two field steps with the source on against the FP64 oracle at the smallest and
largest grid of every segment length (4, 7, 8, 10, 13 and 16 elements on 16
lanes), for slice counts on both sides of the eight XCDs the planes are dealt
to, and for step lengths from one undulator period to 3000 (coefficient r from
below 0.1 to above 10, where a line couples over all its segments instead of
two).  The particle pass is split, so the y sweep also clears the source
behind itself, which the second step would show.  Both sides solve (1 - i r d2)
twice a step; its condition number is sqrt(1 + 16 r^2) and a solve rounds
within about G eps of it, so the fields agree within 4 G eps sqrt(1 + 16 r^2)
a step (MIXED: the field is rounded to FP32 after each sweep, 4 sqrt(1 + 16
r^2) 2^-24), plus the deposition's own error: 1e-13 for the order of its FP64
sums, 2e-5 for MIXED's FP32 terms, the bound of the other field-step tests.
The field records of a run at the same grids cover the sweep with sums."""
from __future__ import annotations

import numpy as np
import pytest

import _oracle
from _oracle import OField, dp, ip
import cases
from cases import LAMBDA0, quad_step
from genesis4_cuda_port_amd import api

pytestmark = pytest.mark.gpu

from test_gpu_parity import gpu_beam, gpu_field, noisy_field, relerr  # noqa: E402


@pytest.mark.parametrize("prec", [api.FP64, api.MIXED])
@pytest.mark.parametrize("periods", [1, 300, 3000])
@pytest.mark.parametrize("ngrid,nslice", [(3, 1), (16, 9), (64, 3), (65, 8), (112, 2), (113, 3),
                                          (128, 9), (129, 1), (160, 2), (161, 3), (208, 2),
                                          (209, 1), (256, 3)])
def test_segment_lengths(ngrid, nslice, periods, prec):
    print(f"case segments ngrid={ngrid} nslice={nslice} periods={periods} prec={prec}", flush=True)
    c = cases.make_case(nslice=nslice, npart=1024, ngrid=ngrid, seed_power=1e6)
    st = quad_step()
    delz = st.delz * periods
    first = nslice // 2
    re, im = noisy_field(c, scale=0.1)
    of = OField(c.nslice, c.ngrid, c.gridmax, LAMBDA0, c.slicelength, 1, re, im, first=first)
    o = c.beam
    r = 0.25 * delz / (2 * np.pi / LAMBDA0 * (2 * c.gridmax / (ngrid - 1)) ** 2)
    eps, dep = (ngrid * 2.0 ** -53, 1e-13) if prec == api.FP64 else (2.0 ** -24, 2e-5)
    with api.Context(0) as ctx:
        f = gpu_field(ctx, c, prec, kind=api.ADI, re=re, im=im, first=first)
        b = gpu_beam(ctx, c, prec)
        for n in (1, 2):
            f.track(b, st, delz)
            sre = np.zeros(c.nslice * ngrid * ngrid)
            sim = np.zeros_like(sre)
            assert _oracle.lib().orc_deposit(c.nslice, ip(o.offsets), dp(o.x), dp(o.y),
                                             dp(o.gamma), dp(o.theta), of.ptr, st, dp(o.current),
                                             delz, dp(sre), dp(sim)) == 1
            _oracle.lib().orc_adi_advance(of.ptr, dp(sre), dp(sim), delz)
            gre, gim, _ = f.download()
            e = relerr(gre + 1j * gim, of.re + 1j * of.im)
            print(f"  step {n} r {r:.3g} rel err {e:.3e}", flush=True)
            assert e < dep + n * 4 * eps * np.sqrt(1 + 16 * r * r)
        f.close()
        b.close()


@pytest.mark.parametrize("prec", [api.FP64, api.MIXED])
@pytest.mark.parametrize("ngrid,nslice", [(3, 1), (64, 3), (65, 8), (112, 2), (113, 3), (128, 9),
                                          (129, 1), (160, 2), (161, 3), (208, 2), (209, 1),
                                          (256, 3)])
def test_segment_length_records(ngrid, nslice, prec):
    """Field records of a three-step run (sums, centre cell, slippage) against
    the oracle's run: each sum within the run tests' bounds (FP64 1e-10, MIXED
    1e-3) of the power times the moment's weight at the grid's edge."""
    print(f"case segment_records ngrid={ngrid} nslice={nslice} prec={prec}", flush=True)
    c = cases.make_case(nslice=nslice, npart=1024, ngrid=ngrid, nsteps=3, seed_power=1e6)
    re, im = noisy_field(c, scale=0.1)
    of = OField(c.nslice, ngrid, c.gridmax, LAMBDA0, c.slicelength, 1, re, im)
    _, _, want = _oracle.run(c.beam, of, c.steps, gamma0=cases.GAMMA0, lambda0=LAMBDA0,
                             solver=api.ADI, sample=c.sample, timerun=c.timerun)
    with api.Context(0) as ctx:
        f = gpu_field(ctx, c, prec, kind=api.ADI, re=re, im=im)
        b = gpu_beam(ctx, c, prec)
        run = api.Run(ctx, b, f, c.steps, LAMBDA0, c.sample, c.timerun, False, 1)
        run.advance(3)
        got = run.download_diag()[1]
        for x in (run, b, f):
            x.close()
    assert got.shape == want.shape
    power = want[:, :, 0].max()
    h = 0.5 * (ngrid - 1)
    amp = np.sqrt(power)
    scale = np.array([power, power * h, power * h * h, power * h, power * h * h, amp * ngrid,
                      amp * ngrid, amp, amp])
    e = np.abs(got - want).max(axis=(0, 1)) / scale
    print(f"  rel err {np.array2string(e, precision=1)}", flush=True)
    assert (e < (1e-10 if prec == api.FP64 else 1e-3)).all()


@pytest.mark.parametrize("prec", [api.FP64, api.MIXED])
@pytest.mark.parametrize("ngrid,bad", [(33, np.nan), (151, np.inf), (255, np.nan), (256, -np.inf)])
def test_non_finite_values_reach_the_whole_plane(ngrid, bad, prec):
    """One value that is not finite in a plane: a single recurrence carries it
    along its row and then along every column, so after one step no cell of
    the plane is finite, and the planes beside it are untouched (the step's own
    bound).  Records say so too."""
    print(f"case segments_non_finite ngrid={ngrid} bad={bad} prec={prec}", flush=True)
    c = cases.make_case(nslice=3, npart=64, ngrid=ngrid, seed_power=1e6, current=0.0)
    st = quad_step()
    plane = ngrid * ngrid
    re, im = noisy_field(c, scale=0.1)
    re[plane + (ngrid // 3) * ngrid + ngrid // 2] = bad
    of = OField(c.nslice, ngrid, c.gridmax, LAMBDA0, c.slicelength, 1, re, im)
    zero = np.zeros_like(re)
    _oracle.lib().orc_adi_advance(of.ptr, dp(zero), dp(zero), st.delz)
    want = (of.re + 1j * of.im).reshape(3, plane)
    assert not np.isfinite(want[1]).any()
    with api.Context(0) as ctx:
        f = gpu_field(ctx, c, prec, kind=api.ADI, re=re, im=im)
        b = gpu_beam(ctx, c, prec)
        f.track(b, st, st.delz)
        gre, gim, _ = f.download()
        power = f.diag_raw()[:, 0]
        f.close()
        b.close()
    got = (gre + 1j * gim).reshape(3, plane)
    assert not np.isfinite(got[1]).any()
    assert list(np.isfinite(power)) == [True, False, True]
    for p in (0, 2):
        assert relerr(got[p], want[p]) < (1e-12 if prec == api.FP64 else 1e-6)


def _wave_totals(v):
    """v [..., 64 lanes] summed as a wave sums it (kernels.hpp wave_total)."""
    lane = np.arange(64)
    for perm in (lane ^ 1, lane ^ 2, lane ^ 7, lane ^ 15):  # the last two: mirrored 8 and 16
        v = v + v[..., perm]
    return (v[..., 0] + v[..., 16]) + (v[..., 32] + v[..., 48])


@pytest.mark.parametrize("ngrid,seg", [(64, 4), (113, 8), (151, 10), (255, 16)])
def test_field_sums_round_as_written(ngrid, seg):
    """The y sweep's field sums, bit for bit: every product and sum rounded on
    its own (no contraction into fused operations), in the order the kernel
    states: the thread's seg rows from the last to the first, the wave, the
    four waves, the 16-column blocks."""
    print(f"case segments_sums ngrid={ngrid}", flush=True)
    c = cases.make_case(nslice=2, npart=64, ngrid=ngrid, seed_power=1e6, current=0.0, nsteps=1)
    re, im = noisy_field(c, scale=0.1)
    with api.Context(0) as ctx:
        f = gpu_field(ctx, c, api.FP64, kind=api.ADI, re=re, im=im)
        b = gpu_beam(ctx, c, api.FP64)
        run = api.Run(ctx, b, f, c.steps, LAMBDA0, c.sample, False, False, 1)
        run.advance(1)
        raw = run.download_diag()[1][1]
        gre, gim, _ = f.download()
        for x in (run, b, f):
            x.close()
    nblk = (ngrid + 15) // 16
    pad = [np.zeros((2, 16 * seg, 16 * nblk)) for _ in range(2)]
    for p, a in zip(pad, (gre, gim)):
        p[:, :ngrid, :ngrid] = a.reshape(2, ngrid, ngrid)
    # [plane, segment, row, block, column]
    r, i = (p.reshape(2, 16, seg, nblk, 16) for p in pad)
    shift = -0.5 * (ngrid - 1)
    wei = r * r + i * i
    dy = (np.arange(16 * seg).reshape(1, 16, seg, 1, 1) + shift)
    terms = [wei, dy * wei, dy * dy * wei, r, i]
    acc = [np.zeros((2, 16, nblk, 16)) for _ in terms]
    for j in range(seg - 1, -1, -1):
        acc = [a + t[:, :, j] for a, t in zip(acc, terms)]
    sw, s3, s4, s5, s6 = acc
    dx = (np.arange(16 * nblk).reshape(1, 1, nblk, 16) + shift)
    for k, a in enumerate((sw, dx * sw, dx * dx * sw, s3, s4, s5, s6)):
        waves = _wave_totals(a.transpose(0, 2, 1, 3).reshape(2, nblk, 4, 64))
        tot = np.zeros(2)
        for blk in range(nblk):
            part = np.zeros(2)
            for w in range(4):
                part = part + waves[:, blk, w]
            tot = tot + part
        assert np.array_equal(tot, raw[:, k]), k
