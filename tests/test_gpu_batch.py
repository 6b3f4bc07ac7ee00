"""GPU: batches of independent steady-state runs (g4h_batch_*).

Each run of a batch (uneven particle counts, two grid sizes, some with an
aw taper) must give the records it gives when run alone through g4h_run
(same kernels, per-slice parameter table instead of by-value parameters),
and one run is checked against the FP64 oracle.

Bars: FP64 1e-12 relative against the lone run and 1e-10 against the
oracle on slice power and bunching; MIXED 1e-6 against the lone MIXED run.
ADI batches run by default as one launch per kernel and step for all runs
(G4H_TUNE_BATCH = 0), and can also run as one launch over all steps (1) or
as per-grid launches on per-grid streams (2); the three must agree to the
same bars (and on particle counts exactly)."""
from __future__ import annotations

import numpy as np
import pytest

import _oracle
from _oracle import OField
from cases import AW, GAMMA0, LAMBDA0, LAMBDAU
from genesis4_cuda_port_amd import api
from genesis4_cuda_port_amd._abi import TUNE_BATCH

pytestmark = pytest.mark.gpu

NSTEPS = 30
GRIDMAX = 0.3e-3


def relerr(a, b):
    den = np.linalg.norm(np.ravel(b))
    return np.linalg.norm(np.ravel(a) - np.ravel(b)) / (den if den > 0 else 1.0)


def _runs():
    taper = AW * (1 - 2e-3 * np.arange(NSTEPS) / NSTEPS - 1e-3 * (np.arange(NSTEPS) / NSTEPS) ** 2)
    base = dict(nbins=4, gridmax=GRIDMAX, current=3000.0, gamma0=GAMMA0, espread_rel=1e-4,
                emitn=0.4e-6, beta=15.0, shotnoise=True, seed_w0=50e-6)
    return [
        dict(base, npart=512, ngrid=33, seed=11, seed_power=1e6),
        dict(base, npart=1024, ngrid=31, seed=12, seed_power=0.0),
        dict(base, npart=512, ngrid=33, seed=13, seed_power=1e5, aw=taper),
        dict(base, npart=256, ngrid=31, seed=14, seed_power=1e6, aw=taper[::-1].copy()),
        dict(base, npart=768, ngrid=33, seed=15, seed_power=0.0, current=1500.0),
    ]


def _steps():
    return api.lattice_fodo(LAMBDAU, [AW], NSTEPS, 10, 3, 1.5, 1)


def _lone(ctx, prec, r, steps):
    beam = api.load_beam(nslice=1, npart=r["npart"], nbins=r["nbins"], gamma0=r["gamma0"],
                         espread_rel=r["espread_rel"], emitn=r["emitn"], beta=r["beta"],
                         slicelength=LAMBDA0, current=r["current"], shotnoise=r["shotnoise"],
                         seed=r["seed"])
    st = api.steps_array(list(steps))
    if r.get("aw") is not None:
        for i in range(len(st)):
            st[i].aw = float(r["aw"][i])
    if r["seed_power"] > 0:
        re, im = api.seed_gaussian(1, r["ngrid"], GRIDMAX, LAMBDA0, r["seed_power"], r["seed_w0"])
    else:
        re = np.zeros(r["ngrid"] ** 2)
        im = np.zeros_like(re)
    return beam, st, re, im


def _power_bunching(braw, fraw, ngrid, current):
    dg = 2 * GRIDMAX / (ngrid - 1)
    P = np.array([api.finalize_field(fraw[k], dg, LAMBDA0, LAMBDA0)[0][0, 0]
                  for k in range(len(fraw))])
    B = np.array([api.finalize_beam(braw[k], 1, [current], GAMMA0)[0][0, 25]
                  for k in range(len(braw))])
    return P, B


@pytest.mark.parametrize("solver", [api.ADI, api.FFT])
@pytest.mark.parametrize("prec", [api.FP64, api.MIXED])
def test_batch_runs_match_lone_runs(gpu_ctx, prec, solver):
    print(f"case batch prec={prec} solver={solver}", flush=True)
    runs = _runs()
    if solver == api.FFT:  # powers of two: the register FFT kernels
        for r in runs:
            r["ngrid"] = {33: 32, 31: 64}[r["ngrid"]]
    steps = _steps()
    batch = api.Batch(gpu_ctx, prec, solver, runs, steps, LAMBDA0)
    assert batch.advance(NSTEPS) == NSTEPS
    assert batch.records() == NSTEPS + 1
    tol = 1e-12 if prec == api.FP64 else 1e-6
    for i, r in enumerate(runs):
        braw, fraw = batch.download(i)
        beam, st, re, im = _lone(gpu_ctx, prec, r, steps)
        b = api.Beam(gpu_ctx, prec, beam.offsets, beam.current, GAMMA0)
        b.upload(beam.x, beam.y, beam.px, beam.py, beam.gamma, beam.theta)
        f = api.Field(gpu_ctx, prec, 1, r["ngrid"], GRIDMAX, LAMBDA0, LAMBDA0)
        f.upload(re, im, 0)
        f.init_solver(solver)
        run = api.Run(gpu_ctx, b, f, st, LAMBDA0, 1.0, False, False, 1)
        run.advance(NSTEPS)
        lb, lf = run.download_diag()
        P, B = _power_bunching(braw[:, None, :], fraw[:, None, :], r["ngrid"], r["current"])
        lP, lB = _power_bunching(lb, lf, r["ngrid"], r["current"])
        ep, eb = relerr(P, lP), relerr(B, lB)
        print(f"  run {i}: power {ep:.3e} bunching {eb:.3e}", flush=True)
        assert ep < tol and eb < tol, i
        if prec == api.FP64 and i == 2:
            of = OField(1, r["ngrid"], GRIDMAX, LAMBDA0, LAMBDA0, 1, re, im)
            _, ob, ofr = _oracle.run(beam, of, st, gamma0=GAMMA0, lambda0=LAMBDA0,
                                     solver=solver, sample=1.0, timerun=False, nharm=1)
            oP, oB = _power_bunching(ob, ofr, r["ngrid"], r["current"])
            assert relerr(P, oP) < 1e-10 and relerr(B, oB) < 1e-10
        run.close()
        f.close()
        b.close()
    batch.close()


@pytest.mark.parametrize("prec", [api.FP64, api.MIXED])
def test_batch_launch_modes_agree(prec):
    print(f"case batch launch modes prec={prec}", flush=True)
    runs = _runs()
    runs.append(dict(runs[0], npart=4096, ngrid=101, seed=16, seed_power=1e5))
    runs.append(dict(runs[1], npart=2048, ngrid=255, seed=17))
    steps = _steps()
    out = {}
    for variant in (0, 1, 2):
        with api.Context(0) as ctx:
            ctx.set_variant(TUNE_BATCH, variant)
            batch = api.Batch(ctx, prec, api.ADI, runs, steps, LAMBDA0)
            # in two pieces: the one-launch path resumes where it stopped
            assert batch.advance(NSTEPS // 2) == NSTEPS // 2
            assert batch.advance(NSTEPS) == NSTEPS
            assert batch.records() == NSTEPS + 1
            out[variant] = [batch.download(i) for i in range(len(runs))]
            batch.close()
    tol = 1e-12 if prec == api.FP64 else 1e-6
    for v in (1, 2):
        for i, r in enumerate(runs):
            (b0, f0), (b1, f1) = out[0][i], out[v][i]
            P0, B0 = _power_bunching(b0[:, None, :], f0[:, None, :], r["ngrid"], r["current"])
            P1, B1 = _power_bunching(b1[:, None, :], f1[:, None, :], r["ngrid"], r["current"])
            ep, eb = relerr(P1, P0), relerr(B1, B0)
            print(f"  variant {v} run {i} (ngrid {r['ngrid']}): power {ep:.3e} bunching {eb:.3e}",
                  flush=True)
            assert ep < tol and eb < tol, (v, i)
            assert np.array_equal(b0[:, 12], b1[:, 12])  # particle counts


@pytest.mark.parametrize("prec", [api.FP64, api.MIXED])
def test_batch_field_records_equal_lone_runs(gpu_ctx, prec):
    """Every number of the field records of 40 runs (more than a workgroup of
    the record kernel takes) on grids of 3 and 9 line blocks.  No current, so
    no deposition: equal bit for bit to lone runs, whose sweeps and sums take
    the same order."""
    print(f"case batch field records prec={prec}", flush=True)
    steps = _steps()
    runs = [dict(npart=64, nbins=4, ngrid=(33, 129)[i % 2], gridmax=GRIDMAX, current=0.0,
                 gamma0=GAMMA0, espread_rel=1e-4, seed=1 + i, seed_power=1e4 * (1 + i),
                 seed_w0=40e-6) for i in range(40)]
    batch = api.Batch(gpu_ctx, prec, api.ADI, runs, steps, LAMBDA0)
    assert batch.advance(NSTEPS) == NSTEPS
    for i in (0, 1, 15, 30, 33, 38, 39):
        r = runs[i]
        _, fraw = batch.download(i)
        g = r["ngrid"]
        re, im = api.seed_gaussian(1, g, GRIDMAX, LAMBDA0, r["seed_power"], r["seed_w0"])
        b = api.Beam(gpu_ctx, prec, np.array([0, 64]), np.zeros(1), GAMMA0)
        z = np.zeros(64)
        b.upload(z, z, z, z, np.full(64, GAMMA0), z)
        f = api.Field(gpu_ctx, prec, 1, g, GRIDMAX, LAMBDA0, LAMBDA0)
        f.upload(re, im, 0)
        f.init_solver(api.ADI)
        run = api.Run(gpu_ctx, b, f, steps, LAMBDA0, 1.0, False, False, 1)
        run.advance(NSTEPS)
        want = run.download_diag()[1][:, 0]
        assert want[:, 0].min() > 0
        assert np.array_equal(fraw, want), i
        for x in (run, f, b):
            x.close()
    batch.close()
