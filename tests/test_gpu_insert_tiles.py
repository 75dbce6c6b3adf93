"""The tiled insertion against the FP32 oracle where its tiles and classes end:
boxes that are and are not multiples of the tile (one tile in all, a last tile of
one or two voxels, the wrapped +-NSAM/2 row in a tile's middle), magnifications
that need two, three and more point classes per axis, axis-aligned planes (three
voxels on an axis at negative integers), more tasks than one listing pass, and an
IRREC that leaves tiles empty.

Bar: every voxel sums at most n = 8 copies x particles x 64 terms, each rounded to
2^-24 of itself, in another order than the oracle: relative L2 below
sqrt(n) 2^-24 x 4 < 1.6e-5 for the largest n here (4,800 per voxel at the origin);
NKSUM and the set of voxels are exact.
"""
import ctypes as C

import numpy as np
import pytest

torch = pytest.importorskip("torch")
import oracle_lib as O  # noqa: E402

pytestmark = pytest.mark.gpu
if not torch.cuda.is_available():  # pragma: no cover
    pytest.skip("no HIP device", allow_module_level=True)

from frealign_amd import api  # noqa: E402

DEV = "cuda"


@pytest.mark.parametrize("nsam,nb,asym,nasym,amag,rrec", [
    (8, 3, "C", 1, (1.0,), 0.5), (16, 4, "D", 2, (1.0, 1.2), 0.5),
    (18, 4, "C", 1, (1.0, 0.6), 0.5), (36, 6, "C", 4, (1.0, 1.17, 0.9), 0.5),
    (50, 5, "C", 1, (2.1, 1.0, 1.16), 0.4), (64, 40, "D", 7, (1.0,), 0.25),
    (90, 3, "O", 1, (1.0, 1.02, 0.97), 0.45), (72, 4, "C", 1, (3.2, 0.8), 0.5)])
@pytest.mark.parametrize("aligned", [False, True])
def test_insert_tiles_vs_oracle(nsam, nb, asym, nasym, amag, rrec, aligned):
    rng = np.random.default_rng(nsam + 7 * aligned)
    jc, nv = nsam // 2 + 1, nsam * nsam * (nsam // 2 + 1)
    cplx = lambda *s: (rng.standard_normal(s) + 1j * rng.standard_normal(s)).astype(np.complex64)  # noqa: E731
    datc, ctff = cplx(nb, nsam, jc), cplx(nb, 2, nsam, jc)
    recb = np.zeros((nb, 10), np.float32)
    recb[:, 0:3] = rng.uniform(-np.pi, np.pi, (nb, 3))
    if aligned:
        recb[:, 0:3] = np.round(recb[:, 0:3] / (np.pi / 2)) * np.float32(np.pi / 2)
    recb[:, 3:5] = rng.uniform(-0.3, 0.3, (nb, 2))
    recb[:, 5] = np.resize(amag, nb)
    recb[:, 6:8] = rng.uniform(0.5, 2.0, (nb, 2))
    recb[:, 8], recb[:, 9] = 0.5, rrec
    half = rng.integers(0, 2, nb).astype(np.int32)
    sym = api.point_group(asym, nasym)
    nsym, symop, jsym, _ = sym
    ctx = api.Context(0)
    outs = []
    for _ in range(2):
        vols = api.HalfMaps.zeros(nsam)
        ctx.insert(nsam, torch.from_numpy(datc).to(DEV), torch.from_numpy(ctff).to(DEV), recb,
                   half, sym, 5.0, 40.0, 1.5, vols)
        outs.append([x.cpu().numpy() for x in (*vols.num, *vols.ctf2, vols.nksum, vols.ttd)])
    ctx.close()
    for a, b in zip(*outs):
        assert np.array_equal(a.view(np.uint8), b.view(np.uint8))
    L = O.oracle()
    for h in range(2):
        num, c2 = np.zeros(nv, np.complex64), np.zeros(nv, np.float32)
        ttd, nk = C.c_double(0), C.c_int64(0)
        for b in np.flatnonzero(half == h):
            r = recb[b]
            on = np.float32(r[6]) / np.float32(r[7])
            L.or32_pinsert(nsam, float(r[9]), float(r[5]), datc[b].reshape(-1),
                           ctff[b].reshape(-1), num, c2, C.byref(ttd), *map(float, r[0:5]),
                           float(r[8]), 5.0, 40.0, nsym, jsym, symop, C.byref(nk), 1.5, float(on),
                           O.IDENTITY, 0)
        got = [outs[0][h].reshape(-1), outs[0][2 + h].reshape(-1)]
        assert outs[0][4][h] == nk.value
        assert np.array_equal(got[1] != 0, c2 != 0)
        for g, w in zip(got, (num, c2)):
            assert np.linalg.norm(g - w) <= 1.6e-5 * np.linalg.norm(w)
        assert abs(outs[0][5][h] - ttd.value) <= 1e-6 * abs(ttd.value)


@pytest.mark.parametrize("nsam", [16, 36])
def test_statistics_phases(nsam):
    """PSUM of one particle on the volume's own grid, a term a voxel: the phase
    difference to the reference on the octants' edges, across the half turn and in
    between, zero where the reference is.  Bar: two arctangents and the result rounded
    to 2^-24 of pi: 4e-7."""
    rng = np.random.default_rng(nsam)
    jc = nsam // 2 + 1

    def phases(*shape):
        a = rng.integers(-8, 9, shape) * np.pi / 8 + rng.choice([0, 0, 1e-6, -1e-6], shape)
        a = np.where(rng.uniform(size=shape) < 0.3, rng.uniform(-np.pi, np.pi, shape), a)
        return (10 ** rng.uniform(-3, 3, shape) * np.exp(1j * a)).astype(np.complex64)

    datc, ref = phases(1, nsam, jc), phases(nsam, nsam, jc)
    axis = np.array([1, -1, 1j, -1j], np.complex64)  # exact axes, with signed zeros
    datc[0, ::3, ::2] = axis[rng.integers(0, 4, datc[0, ::3, ::2].shape)]
    ref[0, ::2, ::3] = -axis[rng.integers(0, 4, ref[0, ::2, ::3].shape)]
    ref[0, 1, ::2] = 0
    ctff = np.zeros((1, 2, nsam, jc), np.complex64)
    ctff[:, 0] = 1
    recb = np.zeros((1, 10), np.float32)
    recb[0, 5:10] = 1, 1, 1, 0.5, 0.45
    ctx = api.Context(0)
    vols = api.HalfMaps.zeros(nsam)
    stats = api.VoxelStats.zeros(nsam, torch.from_numpy(ref).to(DEV))
    ctx.insert(nsam, torch.from_numpy(datc).to(DEV), torch.from_numpy(ctff).to(DEV), recb,
               np.zeros(1, np.int32), api.point_group("C", 1), 5.0, 40.0, 1.5, vols, stats=stats)
    ctx.close()
    j = np.arange(nsam)
    j = np.where(j >= jc, j - nsam, j)
    r2 = j[:, None] ** 2 + np.arange(jc)[None] ** 2
    on = (r2 <= int(nsam * np.float32(0.45)) ** 2) & (r2 > 0)
    d, r = datc[0].astype(np.complex128), ref[0].astype(np.complex128)
    want = np.where(r == 0, 0.0, np.abs(np.angle(d * np.conj(r))))
    got, cnt = stats.psum.cpu().numpy(), stats.ksum.cpu().numpy()
    assert (cnt[0][on] >= 1).all() and on.sum() > 40
    assert np.abs(got[0] - want)[on].max() <= 4e-7
    size = stats.asum.cpu().numpy()[0]
    term = np.abs(vols.num[0].cpu().numpy()[0].astype(np.complex128))
    assert (np.abs(size - term)[on] <= 1e-6 * term[on]).all()
    assert np.abs(got[2:]).max() == 0
