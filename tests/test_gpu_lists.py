"""Several Fields in one launch against the same Fields one by one."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope='module')
def L():
    import lentil_amd
    return lentil_amd


def rel(a, b):
    return float((a - b).norm() / b.norm())


# limits: all in one group; several groups; large ones between small ones; nothing grouped
@pytest.mark.parametrize('one,total', [(1 << 20, 1 << 22), (1 << 20, 9000), (6000, 1 << 22), (10, 10)])
@pytest.mark.parametrize('precision', ['fp32', 'bf16x3'])
def test_dft2_list(L, one, total, precision, monkeypatch):
    monkeypatch.setattr(L.fourier, '_LIST_ONE', one)
    monkeypatch.setattr(L.fourier, '_LIST_ALL', total)
    rng = np.random.default_rng(one + total)
    jobs = []
    for i, (m, n, M, N) in enumerate([(33, 20, 64, 40), (1, 1, 3, 5), (64, 64, 70, 70), (90, 31, 31, 90), (17, 129, 64, 65)]):
        f = torch.from_numpy(rng.standard_normal((m, 2 * n)) + 1j * rng.standard_normal((m, 2 * n))).cuda()
        f = [f, f.to(torch.complex64), f.real.contiguous(), f.real.to(torch.float32), f][i][:, :n]  # rows 2n apart
        jobs.append((f, (1.3 / (m + M), 0.9 / (n + N)), (M, N), (0.4 * i, -0.25), (i, -2)))
    got = L.fourier.dft2_list(jobs, precision=precision)
    for F, (f, alpha, shape, shift, offset) in zip(got, jobs):
        want = L.fourier.dft2(f, alpha, shape, shift, offset, precision=precision)
        assert F.shape == want.shape and F.dtype == torch.complex64
        # two roundings of one transform: bf16 pairs hold 2^-17, FP32 sums 2^-24 per term
        assert rel(F, want) < (2e-5 if precision == 'bf16x3' else 2e-6)


@pytest.mark.parametrize('count', [1, 2, 8, 9, 33, 70])
def test_phasors_and_groups(L, count):
    """Phasors of many segments and their coherent sum (one launch up to 64 Fields, merged above)."""
    rng = np.random.default_rng(count)
    n, wl = 40, 650e-9
    mask = np.zeros((count, n, n))
    for k in range(count):
        r, c = rng.integers(0, n - 9, 2)
        mask[k, r:r + 1 + k % 9, c:c + 2 + k % 7] = 1
    amp, opd = rng.uniform(0.5, 1, (n, n)), rng.normal(0, 1e-7, (n, n))
    pupil = L.Pupil(amplitude=amp, opd=opd, mask=mask, pixelscale=1 / n, focal_length=10.0)
    w = L.Wavefront(wl) * pupil
    ph = amp * np.exp(2j * np.pi * opd / wl)
    assert len(w.data) == count
    for k, f in enumerate(w.data):
        rows, cols = np.nonzero(mask[k])
        want = (ph * mask[k])[rows.min():rows.max() + 1, cols.min():cols.max() + 1]
        assert np.abs(f.data.cpu().numpy() - want).max() < 1e-6    # FP32 phasor
    # every Field moved, clipped and overlapping: |sum|^2 against the host
    shape = (31, 50)
    fields = [L.field.Field(f.data, pixelscale=1.0, offset=(int(a), int(b))) for f, (a, b) in
              zip(w.data, rng.integers(-22, 22, (count, 2)))]
    total = np.zeros(shape)
    for g in L.field._reduce(fields):
        acc = np.zeros((200, 200), complex)
        for f in g['field']:
            r, c = 100 + f.extent[0], 100 + f.extent[2]
            acc[r:r + f.shape[0], c:c + f.shape[1]] += f.data.cpu().numpy()
        total += 0.5 * np.abs(acc[100 - 15:100 + 16, 100 - 25:100 + 25]) ** 2
    for dtype in (torch.float32, torch.float64):
        pitch = torch.full((31, 53), 0.125, dtype=dtype, device='cuda')
        out = L.field.insert_reduced(fields, pitch[:, :50], weight=0.5)
        assert np.abs(out.cpu().numpy() - 0.125 - total).max() < 1e-5 * max(total.max(), 1)
        assert bool((pitch[:, 50:] == 0.125).all())


def test_group_pixelscales_must_agree(L):
    a = torch.ones((8, 8), dtype=torch.complex64, device='cuda')
    fields = [L.field.Field(a, pixelscale=p) for p in (1.0, 2.0)]
    with pytest.raises(ValueError):
        L.field.insert_reduced(fields, torch.zeros((8, 8), device='cuda'))


@pytest.mark.parametrize('bad', [dict(count=65), dict(h=0), dict(ld=3), dict(dtype=0), dict(ldo=5)])
def test_insert_group_refuses(L, bad):
    q = dict(count=1, h=4, ld=4, dtype=1, ldo=8)
    q.update(bad)
    lib, ctx = L._lib.load(), L._lib.context()
    F = torch.ones((4, 4), dtype=torch.complex64, device='cuda')
    out = torch.zeros((8, 8), device='cuda')
    items = (L._lib.MftxField * 65)(*[(F.data_ptr(), q['ld'], q['h'], 4, 0, 0)] * 65)
    assert lib.mftx_insert_group(ctx, items, q['count'], out.data_ptr(), q['dtype'], 8, 8, q['ldo'], 1.0) == L._lib.EINVAL


def test_plan_graph_follows_the_destination(L):
    """Repeating and changing the destination, the type or adding in between gives the same image every
    time, and a call on a stream that is being captured becomes part of that graph."""
    n = 48
    y, x = np.mgrid[:n, :n] / n - 0.5
    pupil = L.Pupil(amplitude=(np.hypot(x, y) < 0.45).astype(float), opd=2e-7 * x * y, pixelscale=1 / n, focal_length=10.0)
    wl = np.linspace(5e-7, 7e-7, 3)
    plan = L.PSFPlan(pupil, wl, None, pixelscale=5e-6, shape=40, oversample=2, precision='fp32')
    want = L.PSFPlan(pupil, wl, None, pixelscale=5e-6, shape=40, oversample=2, precision='fp32', use_graph=False)()
    a, b = torch.empty_like(want), torch.empty_like(want)
    d = torch.empty(want.shape, dtype=torch.float64, device='cuda')
    for dst in (a, a, a, b, a, b, b, b, d, d, d, a, a):
        dst.fill_(float('nan'))
        plan(out=dst)
        assert torch.equal(dst.float(), want)
    plan(out=a, accumulate=True)
    plan(out=a, accumulate=True)
    assert float((a - 3 * want).abs().max()) <= 1e-6 * float(want.max())
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        plan(out=b)
    for _ in range(3):
        b.fill_(float('nan'))
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(b, want)
        plan(out=a)
        assert torch.equal(a, want)
