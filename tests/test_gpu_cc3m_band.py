"""CC3M on the band's own grid against the FFT path on the particle's grid.

The two agree up to FP32 rounding for every box size, band and mask: bands at
the edges of the grids (MAXR2 16 | 17, 24 | 25, 32), boxes smaller than, equal
to and larger than the grid, one item and more items than workgroups, and
items whose AMAG is not 1 (taken by another kernel) between the others.

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
