"""The exhaustive FP32 search with separable shifts against the 225-row product
(the list search over the whole bank in order, which takes it): bands at the edges
of the kernel's forms (16 | 17, 24 | 25, 32 | 33), particle counts that do and do
not fill a quad, and banks of less than one tile and with a short last one.

Bar: a score is a ratio of sums over the band's points, at most 2 x 1,640 products
each rounded to 2^-24 in one order or the other: relative to the largest score
sqrt(3280) 2^-24 x 4 = 1.4e-5.  The views agree where they are further apart.  A
pair's peak, and with it its row and its 3 x 3 box, is the product's also where two
cells of the map tie to a rounding.
"""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu
if not torch.cuda.is_available():  # pragma: no cover
    pytest.skip("no HIP device", allow_module_level=True)

from frealign_amd import api, synth  # noqa: E402

DEV = "cuda"
BAR = 1.4e-5


@pytest.mark.parametrize("nsam,maxr1,maxr2,np_,norient", [
    (64, 1, 16, 1, 40), (72, 0, 17, 3, 40), (96, 2, 24, 4, 300), (100, 2, 25, 5, 68),
    (128, 2, 32, 2, 260), (256, 30, 31, 7, 64), (160, 2, 33, 3, 64), (256, 3, 32, 9, 1028)])
def test_separable_equals_product(nsam, maxr1, maxr2, np_, norient):
    rng = np.random.default_rng(nsam + maxr2)
    jc, k = nsam // 2 + 1, min(32, norient // 4)
    t = lambda a, d: torch.from_numpy(np.ascontiguousarray(a, d)).to(DEV)  # noqa: E731
    vol = t(np.fft.rfftn(rng.standard_normal((nsam,) * 3).astype(np.float32)), np.complex64)
    cplx = lambda *s: rng.standard_normal(s) + 1j * rng.standard_normal(s)  # noqa: E731
    outc, ctff = t(cplx(np_, nsam, jc), np.complex64), t(cplx(np_, 2, nsam, jc), np.complex64)
    dm = t(api.rotation(synth.random_orientations(norient, rng), amag=1.0), np.float32)
    ctx = api.Context(0)
    bank = ctx.search_bank(nsam, maxr1, maxr2, vol, dm, dtype=torch.float32)
    got = ctx.search(nsam, maxr1, maxr2, 0.001, bank, outc, ctff, topk=k, group=4)
    cand = t(np.tile(np.arange(norient), (np_, 1)), np.int32)
    want = ctx.search_list(nsam, maxr1, maxr2, 0.001, bank, outc, ctff, cand, 4, topk=k)
    again = ctx.search(nsam, maxr1, maxr2, 0.001, bank, outc, ctff, topk=k, group=4)
    (o, r, s), (wo, wr, ws) = ([x.cpu().numpy() for x in q] for q in (got, want))
    for a, b in zip(got, again):
        assert torch.equal(a, b)
    ctx.close()
    bar = BAR * np.abs(ws).max()
    assert np.isfinite(s).all() and np.abs(s - ws).max() <= bar
    # (view, shift) agree where the neighbours in the list are not tied to the bar
    gap = np.abs(np.diff(ws, axis=1, prepend=np.inf, append=-np.inf))
    clear = (gap[:, :-1] > 4 * bar) & (gap[:, 1:] > 4 * bar)
    clear[:, -1] = False  # the next one is not in the list
    assert clear.sum() >= 0.7 * clear[:, :-1].size
    assert (o == wo)[clear].all() and (r == wr)[clear].all()


@pytest.mark.parametrize("maxr1,maxr2", [(1, 10), (2, 17), (2, 24)])
def test_tied_peaks_are_the_products(maxr1, maxr2):
    """Particles X1 + c X2 whose maps against one template have two equal cells at the
    top, in 64 bits: the rounding of the sums decides, and the boxes around the two
    differ.  Each row is the product's, each score within the bar."""
    nsam, np_, norient, top = 96, 96, 8, 8
    rng = np.random.default_rng(maxr2)
    jc = nsam // 2 + 1
    t = lambda a, d: torch.from_numpy(np.ascontiguousarray(a, d)).to(DEV)  # noqa: E731
    vol = t(np.fft.rfftn(rng.standard_normal((nsam,) * 3).astype(np.float32)), np.complex64)
    dm = t(api.rotation(synth.random_orientations(norient, rng), amag=1.0), np.float32)
    ctx = api.Context(0)
    bank = ctx.search_bank(nsam, maxr1, maxr2, vol, dm, dtype=torch.float32)
    # the annulus, I-major; the map of ccp.f:194-252 as a matrix over its points
    pts = np.array([(i, j) for i in range(jc - 1) for j in range(1 - jc, jc)
                    if max(1, maxr1 * maxr1) <= i * i + j * j < maxr2 * maxr2])
    s13 = np.stack(np.meshgrid(np.arange(-6, 7), np.arange(-6, 7), indexing="ij"), -1)
    nsamr = 2 * ((nsam // 2 + 1) // 2)
    ph = np.exp(2j * np.pi / nsamr * (s13.reshape(-1, 2) @ pts.T))
    ph *= np.where(pts[:, 0] > 0, 2.0, 1.0)
    tmpl = bank.cpu().numpy().astype(np.float64)[:, :2 * len(pts)]
    tmpl = tmpl[:, ::2] + 1j * tmpl[:, 1::2]
    spec = np.zeros((np_, nsam, jc), np.complex64)
    for p in range(np_):
        m = ph * np.conj(tmpl[p % norient])
        while True:
            x = rng.standard_normal((2, len(pts))) + 1j * rng.standard_normal((2, len(pts)))
            m1, m2 = (m @ x.T).real.T
            a, b = np.argsort(m1)[:-3:-1]
            c = (m1[b] - m1[a]) / (m2[a] - m2[b])
            if set(np.argsort(m1 + c * m2)[-2:]) == {a, b}:
                break
        spec[p, pts[:, 1], pts[:, 0]] = x[0] + c * x[1]
    ctff = np.zeros((np_, 2, nsam, jc), np.complex64)
    ctff[:, 0] = 1.0
    args = (t(spec, np.complex64), t(ctff, np.complex64))
    got = ctx.search(nsam, maxr1, maxr2, 0.0, bank, *args, topk=top, group=1)
    cand = t(np.tile(np.arange(norient), (np_, 1)), np.int32)
    want = ctx.search_list(nsam, maxr1, maxr2, 0.0, bank, *args, cand, 1, topk=top)
    ctx.close()
    (o, r, s), (wo, wr, ws) = ([x.cpu().numpy() for x in q] for q in (got, want))
    bar, seen = BAR * np.abs(ws).max(), 0
    for p in range(np_):
        mine = {k: (a, b) for k, a, b in zip(o[p], r[p], s[p]) if k >= 0}
        for k, a, b in zip(wo[p], wr[p], ws[p]):
            if k >= 0:
                assert mine[k][0] == a and abs(mine[k][1] - b) <= bar, (p, k)
                seen += k == p % norient
    assert seen >= 0.9 * np_  # the tied pairs are in the lists
