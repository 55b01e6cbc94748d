"""Launches of the phase-retrieval tail: the gradient over all OPDs and wavelengths, and the reduction of
partial images into regions of one image."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope='module')
def L():
    import lentil_amd
    return lentil_amd


def rel(a, b):
    return np.linalg.norm(a - b) / np.linalg.norm(b)


# one past and one short of the 8 loads a thread keeps in flight, one OPD and several, every type
@pytest.mark.parametrize('m,n,nw,nd,adt,odt,gdt,with_amp', [
    (1, 1, 1, 1, 'f8', 'f8', 'f8', True), (33, 65, 7, 3, 'f4', 'f8', 'f4', True), (40, 56, 8, 1, 'f8', 'f4', 'f4', False),
    (17, 300, 9, 2, 'f8', 'f8', 'f8', True), (64, 64, 17, 4, 'f4', 'f4', 'f8', False)])
def test_phase_grad_stack(L, m, n, nw, nd, adt, odt, gdt, with_amp):
    rng = np.random.default_rng(m * n + nw)
    amp = rng.uniform(0, 1, (m, n)).astype(adt)
    opd = rng.normal(0, 2e-7, (nd, m, n)).astype(odt)
    wls = np.linspace(500e-9, 800e-9, nw)
    D = (rng.standard_normal((nd, nw, m, n)) + 1j * rng.standard_normal((nd, nw, m, n))).astype(np.complex64)
    lib, ctx = L._lib.load(), L._lib.context()
    ad, od, Dd, iw = (torch.from_numpy(x).cuda() for x in (amp, opd, D, 1 / wls))
    tdt = dict(f4=torch.float32, f8=torch.float64)[gdt]
    # written, not added to: stale values in the outputs must not survive
    g = torch.full((m, n), float('nan'), dtype=tdt, device='cuda')
    ga = torch.full((m, n), float('nan'), dtype=tdt, device='cuda')
    code = L._lib.dtype_code
    L._lib.check(lib.mftx_phase_grad_stack(ctx, ad.data_ptr(), code(ad), n, od.data_ptr(), code(od), n, m * n, nd, m, n,
                                           iw.data_ptr(), nw, Dd.data_ptr(), n, m * n, g.data_ptr(), code(g), n,
                                           ga.data_ptr() if with_amp else None, code(ga), n), ctx, 'stack')
    k = 2 * np.pi / wls[None, :, None, None]
    cd = np.conj(D.astype(complex)) * np.exp(1j * k * opd.astype(float)[:, None])
    ref = np.sum(-2 * k * amp.astype(float) * cd.imag, axis=(0, 1))
    # FP32 phasors (6e-8 relative each) and one rounding of the result
    assert rel(g.cpu().numpy(), ref) < 1e-6
    if with_amp:
        assert rel(ga.cpu().numpy(), np.sum(2 * cd.real, axis=(0, 1))) < 1e-6
    else:
        assert bool(torch.isnan(ga).all())


@pytest.mark.parametrize('bad', [dict(nw=0), dict(nd=0), dict(strideD=1), dict(strideO=1), dict(gdt=0), dict(iw=None)])
def test_phase_grad_stack_refuses(L, bad):
    m = n = 8
    q = dict(nw=2, nd=2, strideD=m * n, strideO=m * n, gdt=3, iw=0)
    q.update(bad)
    lib, ctx = L._lib.load(), L._lib.context()
    z = torch.zeros(4, m, n, dtype=torch.complex64, device='cuda')
    d = torch.ones(2, m, n, dtype=torch.float64, device='cuda')
    rc = lib.mftx_phase_grad_stack(ctx, d.data_ptr(), 3, n, d.data_ptr(), 3, n, q['strideO'], q['nd'], m, n,
                                   None if q['iw'] is None else d.data_ptr(), q['nw'], z.data_ptr(), n, q['strideD'],
                                   d.data_ptr(), q['gdt'], n, None, 3, n)
    assert rc == L._lib.EINVAL


# images whose regions overlap, differ per wavelength, leave pixels uncovered or stick out; row strides; adding
@pytest.mark.parametrize('accumulate', [False, True])
@pytest.mark.parametrize('dtype', [torch.float32, torch.float64])
@pytest.mark.parametrize('shape,prop,copies,tilt', [((40, 40), None, 1, (0, 0)), ((37, 130), (20, 24), 1, (3.0, -9.0)),
                                                    ((65, 33), (30, 30), 3, (-20.0, 8.0)), ((30, 30), None, 2, (400.0, 0))])
def test_reduce_regions(L, shape, prop, copies, tilt, dtype, accumulate):
    n, os, du, z = 48, 2, 5e-6, 10.0
    y, x = np.mgrid[:n, :n] - n / 2 + 0.5
    amp = (np.hypot(x, y) < n / 2.2).astype(float)
    opd = 60e-9 * np.sin(x / 7) * np.cos(y / 5)
    wls = np.linspace(500e-9, 750e-9, 5)
    pupil = L.Pupil(amplitude=amp, opd=opd, mask=np.ones((n, n)), pixelscale=1 / n, focal_length=z)
    tilts = [L.Tilt(*(t * du / os / z for t in tilt))]
    # a dispersed spot: every wavelength has its own window
    tilts.append(L.DispersiveTilt(trace=[0.5, 0], dispersion=[5e-9 / du, 600e-9]))
    plan = L.PSFPlan(pupil, wls, np.full(5, 0.2), pixelscale=du, shape=shape, prop_shape=prop, oversample=os,
                     tilts=tilts, precision='fp32', copies=copies, use_graph=False)
    rows, cols = plan.shape_out
    pitch = torch.full((rows, cols + 3), 0.25 if accumulate else float('nan'), dtype=dtype, device='cuda')
    got = plan(out=pitch[:, :cols], accumulate=accumulate).cpu().numpy()
    want = np.zeros((rows, cols // copies))
    for wl in wls:
        w = L.Wavefront(wl) * pupil
        for t in tilts:
            w = w * t
        w = L.propagate_dft(w, pixelscale=du, shape=shape, prop_shape=prop, oversample=os, precision='fp32')
        want = w.insert(want, weight=0.2)
    want = np.tile(want, (1, copies)) + (0.25 if accumulate else 0)
    # both sum the same FP32 fields; 2^-24 of the sum per rounding, 2e-6 of the peak for the transforms
    assert np.abs(got - want).max() <= 4e-6 * max(np.abs(want).max(), 1e-6)
    assert bool(torch.isnan(pitch[:, cols:]).all()) != accumulate
