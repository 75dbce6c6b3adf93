"""CC3M on the band's own grid against the FFT path on the particle's grid.

The two agree up to FP32 rounding for every box size, band and mask, and an item's
score has the same bits whatever the other items of its call are: bands at
the edges of the grids (MAXR2 16 | 17, 24 | 25, 32), boxes smaller than, equal
to and larger than the grid, one item and more items than workgroups, and
items whose AMAG is not 1 (taken by another kernel) between the others.  The
window form is held to the scores at its shifts in the same way.

Bar: both paths run about 2 log2(N^2) + 4 rounded stages (transforms, mask,
shell sums), each at most 2^-24 of the shells' root mean square, so a score
moves by no more than about 40 x 2^-24 x sqrt(shells) = 1.4e-5 of the largest.
"""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu
if not torch.cuda.is_available():  # pragma: no cover
    pytest.skip("no HIP device", allow_module_level=True)

from frealign_amd import _native as N  # noqa: E402
from frealign_amd import api, synth  # noqa: E402

DEV = "cuda"
BAR = 1.4e-5


@pytest.fixture(scope="module")
def ctx():
    c = (api.Context(0), api.Context(0))  # the default launch, and the FFT path
    yield c
    for x in c:
        x.close()


def items(nsam, npart, n, seed, mags):
    rng = np.random.default_rng(seed)
    jc = nsam // 2 + 1
    t = lambda a, d=np.float32: torch.from_numpy(np.ascontiguousarray(a, d)).to(DEV)  # noqa: E731
    vol = np.fft.rfftn(rng.standard_normal((nsam,) * 3).astype(np.float32))
    spec = np.fft.rfft2(rng.standard_normal((npart, nsam, nsam)))
    ctff = rng.standard_normal((npart, 2, nsam, jc)) + 1j * rng.standard_normal((npart, 2, nsam, jc))
    amag = np.where(rng.uniform(size=n) < 0.3, 1.04, 1.0) if mags else np.ones(n)
    dm = api.rotation(synth.random_orientations(n, rng), amag=1.0) / amag[:, None]
    return (t(vol, np.complex64), t(spec, np.complex64), t(ctff, np.complex64),
            t(np.sort(rng.integers(0, npart, n)), np.int32), t(dm), t(rng.normal(0, 0.1, (n, 2))),
            t(amag))


def score(ctx, nsam, a, maxr1, maxr2, ring, cc3):
    fsct = torch.linspace(1.0, 0.5, nsam // 2 + 1, device=DEV)
    vol, spec, ctff, pidx, dm, shift, amag = a
    out = torch.full((pidx.numel(),), float("nan"), device=DEV)
    ctx._sync_stream()
    fn = N.lib().fr_cc3_batch if cc3 else N.lib().fr_cc3m_batch
    N.check(fn(ctx.h, nsam, pidx.numel(), *(x.data_ptr() for x in a), maxr1, maxr2, 0.002,
               fsct.data_ptr(), ring.ctypes.data, out.data_ptr()), "cc3")
    return out.cpu().numpy()


@pytest.mark.parametrize("nsam,maxr1,maxr2", [
    (64, 0, 16), (64, 2, 17), (64, 1, 31), (96, 1, 16), (96, 2, 24), (96, 2, 25), (96, 0, 32),
    (128, 2, 15), (128, 2, 24), (128, 1, 32), (160, 3, 17), (192, 2, 25), (256, 0, 16),
    (256, 2, 24), (256, 2, 32), (256, 30, 31)])
@pytest.mark.parametrize("cc3", [False, True])
def test_band_grid_equals_fft_path(ctx, nsam, maxr1, maxr2, cc3):
    ri = 0.42 * nsam
    for n, halfw, mags in ((1, 6.0, False), (37, 6.0, True), (1100, 1.0, True)):
        ring = np.array([(ri - halfw / 2) ** 2, (ri + halfw / 2) ** 2, ri - halfw / 2, halfw],
                        np.float32)
        a = items(nsam, min(n, 5), n, 17 * nsam + maxr2 + n, mags)
        ctx[1].set_cc3m_variant(nsam, False)
        want = score(ctx[1], nsam, a, maxr1, maxr2, ring, cc3)
        got = score(ctx[0], nsam, a, maxr1, maxr2, ring, cc3)
        assert np.isfinite(got).all()
        assert np.abs(got - want).max() <= BAR * np.abs(want).max(), (n, halfw)
        again = score(ctx[0], nsam, a, maxr1, maxr2, ring, cc3)
        assert np.array_equal(got, again)


@pytest.mark.parametrize("nsam,maxr1,maxr2,nsh", [
    (64, 1, 16, 0), (64, 2, 31, 2), (96, 0, 24, 3), (96, 2, 25, 4), (128, 2, 32, 5),
    (160, 2, 14, 1), (256, 1, 32, 4)])
@pytest.mark.parametrize("amag", [1.0, 1.04])
def test_window_equals_scores_at_its_shifts(ctx, nsam, maxr1, maxr2, nsh, amag):
    """Each orientation's best score over the window and its shift, against CC3M at
    every shift (one, two and three column blocks of the quarter window)."""
    npart, nang, dang, dsh = 3, 1, 0.02, float(np.float32(2 * np.pi / nsam))
    ri = 0.42 * nsam
    ring = np.array([(ri - 3) ** 2, (ri + 3) ** 2, ri - 3, 6.0], np.float32)
    a3df, spec, ctff = items(nsam, npart, npart, 5 + nsam, False)[:3]
    fsct = torch.linspace(1.0, 0.5, nsam // 2 + 1, device=DEV)
    rng = np.random.default_rng(nsh)
    par = np.concatenate([synth.random_orientations(npart, rng), rng.normal(0, 0.1, (npart, 2))], 1)
    par = par.astype(np.float32)
    best, sc, code = ctx[0].local_search(
        nsam, a3df, spec, ctff, par, nang=nang, dang=dang, nsh=nsh, dsh=dsh, maxr1=maxr1,
        maxr2=maxr2, rbfact=0.002, fsct=fsct, ring=ring, amag=np.full(npart, amag),
        all_scores=True)
    k = np.arange(-nang, nang + 1, dtype=np.float32) * np.float32(dang)
    q = np.arange(-nsh, nsh + 1, dtype=np.float32) * np.float32(dsh)
    ang = np.stack(np.meshgrid(k, k, k, indexing="ij"), -1).reshape(-1, 3)
    sh = np.stack(np.meshgrid(q, q, indexing="ij"), -1).reshape(-1, 2)
    eul = (par[:, None, :3] + ang[None]).reshape(-1, 3)
    n, ns = len(eul), len(sh)
    dm = np.repeat(api.rotation(eul, amag=amag), ns, 0)
    shift = (np.repeat(par[:, 3:], len(ang), 0)[:, None] + sh[None]).reshape(-1, 2)
    t = lambda a, d: torch.from_numpy(np.ascontiguousarray(a, d)).to(DEV)  # noqa: E731
    ctx[1].set_cc3m_variant(nsam, False)
    want = ctx[1].cc3m(nsam, a3df, spec, ctff,
                       t(np.repeat(np.arange(npart), len(ang) * ns), np.int32), t(dm, np.float32),
                       t(shift, np.float32), torch.full((n * ns,), amag, device=DEV), maxr1, maxr2,
                       0.002, fsct, ring).cpu().numpy().reshape(n, ns)
    sc, code = sc.cpu().numpy().reshape(-1), code.cpu().numpy().reshape(-1)
    bar = BAR * np.abs(want).max()
    assert np.abs(sc - want.max(1)).max() <= bar
    assert (want.max(1) - want[np.arange(n), code] <= 2 * bar).all()
    assert np.abs(best[:, 5] - want.reshape(npart, -1).max(1)).max() <= bar


@pytest.mark.parametrize("nsam,maxr1,maxr2", [(36, 1, 16), (72, 0, 32), (100, 2, 25), (250, 2, 32),
                                              (300, 3, 24), (384, 1, 31)])
def test_band_grid_serves_any_box(ctx, nsam, maxr1, maxr2):
    """Candidates of a search (AMAG = 1 throughout) at boxes that the products on the
    particle's grid do not hold, smaller and larger than the band's grid."""
    npart, k, nbank = 3, 5, 40
    rng = np.random.default_rng(nsam)
    ri = 0.42 * nsam
    ring = np.array([(ri - 3) ** 2, (ri + 3) ** 2, ri - 3, 6.0], np.float32)
    vol, spec, ctff, _, dm, _, _ = items(nsam, npart, nbank, nsam, False)
    t = lambda a, d: torch.from_numpy(np.ascontiguousarray(a, d)).to(DEV)  # noqa: E731
    o, row = rng.integers(0, nbank, (npart, k)), rng.integers(0, 225, (npart, k))
    nsamr = 2 * ((nsam // 2 + 1) // 2)
    fsct = torch.linspace(1.0, 0.5, nsam // 2 + 1, device=DEV)
    ctx[1].set_cc3m_variant(nsam, False)
    got, _ = ctx[0].rescore(nsam, vol, spec, ctff, t(o, np.int32), t(row, np.int32),
                            dm.reshape(nbank, 9), nsamr, maxr1, maxr2, 0.002, fsct, ring)
    sh = np.stack([row // 15 - 7, row % 15 - 7], -1).astype(np.float32)
    sh = sh / np.float32(nsamr) * np.float32(2 * 3.1415926535897)
    want = ctx[1].cc3m(nsam, vol, spec, ctff, t(np.repeat(np.arange(npart), k), np.int32),
                       dm.reshape(nbank, 9)[t(o.reshape(-1), np.int64)].contiguous(),
                       t(sh.reshape(-1, 2), np.float32), torch.ones(npart * k, device=DEV), maxr1,
                       maxr2, 0.002, fsct, ring).reshape(npart, k)
    assert (got - want).abs().max() <= BAR * want.abs().max()
    ctx[1].set_cc3m_variant(nsam, True)  # the score entry takes the same way
    same = ctx[1].cc3m(nsam, vol, spec, ctff, t(np.repeat(np.arange(npart), k), np.int32),
                       dm.reshape(nbank, 9)[t(o.reshape(-1), np.int64)].contiguous(),
                       t(sh.reshape(-1, 2), np.float32), torch.ones(npart * k, device=DEV), maxr1,
                       maxr2, 0.002, fsct, ring).reshape(npart, k)
    assert torch.equal(got, same)


def mask(nsam):
    ri = 0.42 * nsam
    return np.array([(ri - 3) ** 2, (ri + 3) ** 2, ri - 3, 6.0], np.float32)


@pytest.mark.parametrize("nsam,maxr1,maxr2", [(36, 1, 16), (72, 0, 32), (100, 2, 25), (128, 2, 24),
                                              (250, 2, 16)])
@pytest.mark.parametrize("cc3", [False, True])
def test_a_score_does_not_depend_on_the_other_items(ctx, nsam, maxr1, maxr2, cc3):
    """Items with AMAG 1 and 1.04 in one call, against each kind and each item by
    itself: the same bits, and all against the particle's grid."""
    a = items(nsam, 3, 40, nsam, True)
    amag = a[-1].cpu().numpy()
    whole = score(ctx[0], nsam, a, maxr1, maxr2, mask(nsam), cc3)
    few = [[k] for k in (0, 1, 2, 39)] + [np.flatnonzero(amag == 1), np.flatnonzero(amag != 1)]
    assert all(len(k) for k in few)
    for k in few:
        idx = torch.as_tensor(np.asarray(k), device=DEV)
        part = a[:3] + tuple(x[idx].contiguous() for x in a[3:])
        assert np.array_equal(score(ctx[0], nsam, part, maxr1, maxr2, mask(nsam), cc3), whole[k])
    if not cc3:  # the checked entry knows which items there are
        fsct = torch.linspace(1.0, 0.5, nsam // 2 + 1, device=DEV)
        got = ctx[0].cc3m(nsam, *a, maxr1, maxr2, 0.002, fsct, mask(nsam)).cpu().numpy()
        assert np.array_equal(got, whole)
    ctx[1].set_cc3m_variant(nsam, False)
    want = score(ctx[1], nsam, a, maxr1, maxr2, mask(nsam), cc3)
    assert np.abs(whole - want).max() <= BAR * np.abs(want).max()


@pytest.mark.parametrize("nsam,maxr2", [(72, 32), (100, 25), (128, 24)])
def test_refinement_does_not_depend_on_the_other_particles(ctx, nsam, maxr2):
    """PREFINE of AMAG 1, 1.04, 1 together and one by one: the same bits."""
    n = 3
    a3df, spec, ctff = items(nsam, n, n, 7 * nsam, False)[:3]
    fsct = torch.linspace(1.0, 0.5, nsam // 2 + 1, device=DEV)
    rng = np.random.default_rng(nsam)
    par = np.zeros((n, 6), np.float32)
    par[:, :3], par[:, 3:5] = synth.random_orientations(n, rng), rng.normal(0, 0.05, (n, 2))
    prior = np.tile(np.array([0, 0, 0.3, 0.3, 0.01], np.float32), (n, 1))
    amag = np.array([1.0, 1.04, 1.0], np.float32)

    def refine(k, free):
        return ctx[0].refine(nsam, a3df, spec, ctff, np.asarray(k, np.int32), amag[k], par[k],
                             np.full(5, free, np.int32), 2, maxr2, 0.0, fsct, mask(nsam), prior[k])

    for free in (1, 0):  # 0: nothing to refine, PRESA alone
        whole, nev = refine([0, 1, 2], free)
        assert not free or len(set(nev.tolist())) > 1  # not all converge in the same round
        for k in range(n):
            got, ne = refine([k], free)
            assert ne[0] == nev[k]
            assert np.array_equal(got[0].view(np.int32), whole[k].view(np.int32))


def test_local_search_does_not_depend_on_the_other_particles(ctx):
    """Particles with AMAG 1, 1.04, 1, -1 together and one by one: the same bits."""
    nsam, maxr2, n = 128, 25, 4
    a3df, spec, ctff = items(nsam, n, n, 3, False)[:3]
    fsct = torch.linspace(1.0, 0.5, nsam // 2 + 1, device=DEV)
    rng = np.random.default_rng(11)
    par = np.concatenate([synth.random_orientations(n, rng), rng.normal(0, 0.1, (n, 2))],
                         1).astype(np.float32)
    amag = np.array([1.0, 1.04, 1.0, -1.0], np.float32)

    def search(k):
        return ctx[0].local_search(nsam, a3df, spec[k].contiguous(), ctff[k].contiguous(), par[k],
                                   nang=1, dang=0.02, nsh=4, dsh=float(np.float32(2 * np.pi / nsam)),
                                   maxr1=2, maxr2=maxr2, rbfact=0.002, fsct=fsct, ring=mask(nsam),
                                   amag=amag[k], all_scores=True)

    best, sc, code = search([0, 1, 2, 3])
    for k in range(n):
        b, s, c = search([k])
        assert np.array_equal(b[0].view(np.int32), best[k].view(np.int32))
        assert torch.equal(s.reshape(-1), sc.reshape(n, -1)[k])
        assert torch.equal(c.reshape(-1), code.reshape(n, -1)[k])


def test_local_search_of_more_orientations_than_one_launch_holds(ctx):
    """15,625 orientations: the cross spectra go through their buffer in two parts.
    The orientations of a smaller grid about the same centre keep their bits."""
    nsam, maxr2 = 64, 31
    a3df, spec, ctff = items(nsam, 1, 1, 4, False)[:3]
    fsct = torch.linspace(1.0, 0.5, nsam // 2 + 1, device=DEV)
    par = np.array([[0.3, 0.8, -0.4, 0.02, -0.01]], np.float32)
    out = {}
    for nang in (2, 12):
        _, s, c = ctx[0].local_search(nsam, a3df, spec, ctff, par, nang=nang, dang=0.02, nsh=2,
                                      dsh=0.1, maxr1=1, maxr2=maxr2, rbfact=0.002, fsct=fsct,
                                      ring=mask(nsam), all_scores=True)
        m, w = 2 * nang + 1, slice(nang - 2, nang + 3)
        out[nang] = (s.reshape(m, m, m)[w, w, w], c.reshape(m, m, m)[w, w, w])
        assert torch.isfinite(s).all()
    assert torch.equal(out[2][0], out[12][0]) and torch.equal(out[2][1], out[12][1])


def test_boxes_beyond_the_largest_are_refused(ctx):
    """CC3M holds boxes up to 516: a rescoring of a larger one is refused whatever
    its band, as a score of it is."""
    nsam, k = 540, 2
    jc = nsam // 2 + 1
    z = lambda *s: torch.zeros(s, dtype=torch.complex64, device=DEV)  # noqa: E731
    vol, spec, ctff = z(nsam, nsam, jc), z(1, nsam, jc), z(1, 2, nsam, jc)
    o = torch.zeros((1, k), dtype=torch.int32, device=DEV)
    dm = torch.from_numpy(api.rotation(np.zeros((1, 3), np.float32), amag=1.0)).to(DEV)
    fsct = torch.ones(jc, device=DEV)
    with pytest.raises(N.NativeError, match="box too large"):
        ctx[0].cc3m(nsam, vol, spec, ctff, o[0, :1].contiguous(), dm, torch.zeros((1, 2), device=DEV),
                    torch.ones(1, device=DEV), 2, 20, 0.0, fsct, mask(nsam))
    with pytest.raises(N.NativeError, match="box too large"):
        ctx[0].rescore(nsam, vol, spec, ctff, o, o + 112, dm, 270, 2, 20, 0.0, fsct, mask(nsam))
