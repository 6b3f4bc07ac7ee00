"""GPU: spectral line steps by pairs of transforms at the edges of their sizes.

Two deposition + FFT steps against the FP64 oracle at the smallest and largest
grids of each transform size (4, 16, 64, 128 and 256 points) and at the first
grid beyond them, for slice counts on both sides of the eight XCDs that the
planes are dealt to.  The particle pass is split (few slices), so the column pass also
clears the source behind itself, which the second step would show.  Bounds of
the other spectral field-step tests: FP64 1e-12, MIXED 2e-5."""
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


@pytest.mark.parametrize("prec,tol", [(api.FP64, 1e-12), (api.MIXED, 2e-5)])
@pytest.mark.parametrize("filtered", [False, True])
@pytest.mark.parametrize("ngrid,nslice", [(3, 1), (15, 9), (17, 9), (31, 3), (33, 9), (63, 8), (65, 1),
                                          (127, 3), (129, 9), (255, 2), (257, 2)])
def test_line_pairs(ngrid, nslice, filtered, prec, tol):
    print(f"case fft lines ngrid={ngrid} nslice={nslice} filter={filtered} prec={prec}", flush=True)
    c = cases.make_case(nslice=nslice, npart=1024, ngrid=ngrid, seed_power=1e6)
    st = quad_step()
    first = nslice // 2
    re, im = noisy_field(c, scale=0.1)
    of = OField(c.nslice, c.ngrid, c.gridmax, LAMBDA0, c.slicelength, 1, re, im, first=first)
    o = c.beam
    plane = ngrid * ngrid
    with api.Context(0) as ctx:
        f = gpu_field(ctx, c, prec, kind=api.FFT, re=re, im=im, first=first)
        f.init_solver(api.FFT, filtered, 0.6, 0.6, 0.1)
        b = gpu_beam(ctx, c, prec)
        for it in range(2):
            f.track(b, st, st.delz)
            sre = np.zeros(c.nslice * plane)
            sim = np.zeros_like(sre)
            assert _oracle.lib().orc_deposit(c.nslice, ip(o.offsets), dp(o.x), dp(o.y),
                                             dp(o.gamma), dp(o.theta), of.ptr, st, dp(o.current),
                                             st.delz, dp(sre), dp(sim)) == 1
            _oracle.lib().orc_fft_advance(of.ptr, dp(sre), dp(sim), st.delz, int(filtered), 0.6,
                                          0.6, 0.1)
            gre, gim, _ = f.download()
            e = relerr(gre + 1j * gim, of.re + 1j * of.im)
            print(f"  step {it}: rel err {e:.3e}", flush=True)
            assert e < tol
        f.close()
        b.close()
