"""CC3M, CC3 and PRESB on the particle's grid against the oracle in 64 bits: lengths
that are and are not compiled in (72, 100, 250), bands from a few columns to the
whole half-plane and not multiples of the column block, magnifications whose ring
mean takes its own pass next to AMAG = 1, an empty ring, and more items than one
launch of the band holds (the same bits as one by one).

Bar: about 2 log2(N^2) + 4 rounded stages between a section and its shell sums, each
2^-24 of the shells' root mean square, FP32 CTF and phases: 40 x 2^-24 x sqrt(shells)
= 3e-5 of the largest score at 160 shells.
"""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
import oracle_lib as O  # noqa: E402

pytestmark = pytest.mark.gpu
if not torch.cuda.is_available():  # pragma: no cover
    pytest.skip("no HIP device", allow_module_level=True)

from frealign_amd import _native as N  # noqa: E402
from frealign_amd import api, synth  # noqa: E402

DEV = "cuda"
BAR = 3e-5


@pytest.fixture(scope="module")
def ctx():
    c = api.Context(0)
    yield c
    c.close()


def case(nsam, n, seed, amag):
    rng = np.random.default_rng(seed)
    jc = nsam // 2 + 1
    vol = np.fft.rfftn(rng.standard_normal((nsam,) * 3).astype(np.float32)).astype(np.complex64)
    spec = np.fft.rfft2(rng.standard_normal((2, nsam, nsam))).astype(np.complex64)
    ctff = (rng.standard_normal((2, 2, nsam, jc))
            + 1j * rng.standard_normal((2, 2, nsam, jc))).astype(np.complex64)
    eul = synth.random_orientations(n, rng)
    am = np.resize(np.asarray(amag, np.float32), n)
    dm = np.concatenate([api.rotation(eul[k:k + 1], amag=float(am[k])) for k in range(n)])
    shift = rng.normal(0, 0.1, (n, 2)).astype(np.float32)
    return vol, spec, ctff, (np.arange(n) % 2).astype(np.int32), eul, am, dm, shift


@pytest.mark.parametrize("nsam,maxr1,maxr2,halfw", [
    (16, 0, 7, 2.0), (72, 1, 35, 6.0), (96, 3, 41, 6.0), (100, 0, 49, 1.0), (128, 2, 33, 6.0),
    (160, 2, 79, 0.0), (250, 70, 71, 6.0), (320, 2, 80, 6.0)])
@pytest.mark.parametrize("cc3", [False, True])
def test_scores_and_presb_vs_oracle(ctx, nsam, maxr1, maxr2, halfw, cc3):
    n, h = 3, nsam // 2
    vol, spec, ctff, pidx, eul, am, dm, shift = case(nsam, n, nsam + maxr2, (1.0, 1.05, 1.1))
    ri = 0.4 * nsam
    ring = np.array([(ri - halfw / 2) ** 2, (ri + halfw / 2) ** 2, ri - halfw / 2, halfw or 1.0],
                    np.float32)
    if halfw == 0.0:
        ring[1] = ring[0]  # no pixel in the ring
    fsct = np.linspace(1.0, 0.5, h + 1).astype(np.float32)
    t = [torch.from_numpy(x).to(DEV) for x in (vol, spec, ctff, pidx, dm, shift, am)]
    fs = torch.from_numpy(fsct).to(DEV)
    out = torch.empty(n, device=DEV)
    ctx.set_cc3m_variant(nsam, False)
    ctx._sync_stream()
    fn = N.lib().fr_cc3_batch if cc3 else N.lib().fr_cc3m_batch
    N.check(fn(ctx.h, nsam, n, *(x.data_ptr() for x in t), maxr1, maxr2, 0.001, fs.data_ptr(),
               ring.ctypes.data, out.data_ptr()), "cc3m")
    rbin = None
    if not cc3 and halfw:
        rbin = ctx.presb(nsam, *t, ring, rbin=torch.full((n, nsam), 7.0, device=DEV))
        rbin = rbin.cpu().numpy()
    L = O.oracle()
    want = np.zeros(n)
    for k in range(n):
        sp, cf = (np.ascontiguousarray(a[pidx[k]], np.complex128).reshape(-1) for a in (spec, ctff))
        pose = [*map(float, eul[k]), *map(float, shift[k])]
        rg = [float(v) for v in ring]
        args = [nsam, float(am[k]), sp, vol.reshape(-1), maxr1, maxr2, *pose, 0.001]
        want[k] = (L.or64_cc3(*args, cf, *rg, O.IDENTITY) if cc3
                   else L.or64_cc3m(*args, fsct, cf, *rg, O.IDENTITY))
        if rbin is not None:
            rb = np.full(nsam, 7.0)
            L.or64_presb(nsam, float(am[k]), sp, vol.reshape(-1), *pose, rb, cf, *rg, O.IDENTITY)
            assert np.abs(rbin[k] - rb).max() <= BAR
    assert np.abs(out.cpu().numpy() - want).max() <= BAR * np.abs(want).max()


def test_chunks_have_the_same_bits(ctx):
    nsam, n, maxr2 = 384, 400, 190  # about 320 items fit one launch's band
    vol, spec, ctff, pidx, eul, am, dm, shift = case(nsam, n, 5, (1.0, 1.0, 1.02))
    ring = np.array([140.0 ** 2, 146.0 ** 2, 140.0, 6.0], np.float32)
    fs = torch.full((nsam // 2 + 1,), 0.5, device=DEV)
    dev = [torch.from_numpy(x).to(DEV) for x in (vol, spec, ctff)]
    per = [torch.from_numpy(x).to(DEV) for x in (pidx, dm, shift, am)]
    run = lambda s: ctx.cc3m(nsam, *dev, *(x[s].contiguous() for x in per), 1, maxr2, 0.0,  # noqa: E731
                             fs, ring)
    whole = run(slice(0, n))
    assert torch.isfinite(whole).all()
    for s in (slice(0, 3), slice(318, 330), slice(397, 400)):
        assert torch.equal(run(s), whole[s])
