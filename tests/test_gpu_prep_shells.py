"""PWEIGHT's shells summed per column block, and the CTF table formed with the
weights: against the oracle without the CTF in the weights (its branch of the
new kernel), and for more images than one round of the shells' scratch holds.

Bar: as for CTFAPPLY's outputs (tests/test_gpu_parity.py), 1e-5 relative L2 of
the FP32 oracle: FP32 transforms of the same length and FP32 sums of at most a
few hundred positive terms, a rounding apart.  A repeated image gives its bits
again wherever it lies in the batch.
"""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
import oracle_lib as O  # noqa: E402

pytestmark = pytest.mark.gpu
if not torch.cuda.is_available():  # pragma: no cover
    pytest.skip("no HIP device", allow_module_level=True)

from frealign_amd import api, synth  # noqa: E402


def _inputs(nsam, nb, rng):
    jc = nsam // 2 + 1
    r = 0.4 * nsam
    # CS, WL, WGH1, WGH2, THETATR, RIH, HALFW, RI2, RI3, TX, TY
    g = np.array([2.7e7, 0.0197, 0.995, 0.1, 0.0197 / nsam, r - 3, 6.0, (r - 3) ** 2, (r + 3) ** 2,
                  0.0, 0.0], np.float32)
    ps = np.linspace(8.0, 0.05, jc + 1).astype(np.float32)
    buf = np.zeros((nb, nsam, nsam + 2), np.float32)
    buf[:, :, :nsam] = rng.standard_normal((nb, nsam, nsam))
    ppar = np.zeros((nb, 8), np.float32)
    ppar[:, 0:2] = rng.uniform(-0.3, 0.3, (nb, 2))
    ppar[:, 2] = rng.uniform(10000, 20000, nb)
    ppar[:, 3] = ppar[:, 2] + rng.uniform(0, 500, nb)
    ppar[:, 5] = 1.0
    return g, ps, buf, ppar


@pytest.mark.parametrize("nsam", [64, 72, 80, 90, 128, 162, 200, 250, 256, 432, 500, 512])
@pytest.mark.parametrize("ictf", [0, 1])
def test_outc_vs_oracle(nsam, ictf):
    rng = np.random.default_rng(nsam + ictf)
    nb, jc = 2, nsam // 2 + 1
    g, ps, buf, ppar = _inputs(nsam, nb, rng)
    ctx = api.Context(0)
    got = ctx.ctfapply(nsam, torch.from_numpy(buf.copy()).cuda(), torch.from_numpy(ppar).cuda(),
                       torch.from_numpy(ps).cuda(), g, ictf)
    L = O.oracle()
    for b in range(nb):
        spec = buf[b].copy().reshape(-1)
        L.or_rfft2_f(nsam, spec)
        want = [np.zeros(k * nsam * jc, np.complex64) for k in (2, 1, 1)]
        L.or32_ctfapply(nsam, spec.view(np.complex64).copy(), *[float(x) for x in ppar[b, :2]],
                        *[float(x) for x in g[:4]], *[float(x) for x in ppar[b, 2:5]], float(g[4]),
                        float(ppar[b, 5]), *[float(x) for x in g[5:9]], ps, ictf, *want)
        for x, y in zip(got, want):
            x = x[b].cpu().numpy().reshape(-1)
            assert np.linalg.norm(x - y) < 1e-5 * np.linalg.norm(y)
    ctx.close()


def test_more_images_than_a_round():
    """49,056 images of a 64 box fill the shells' 32 MB."""
    rng = np.random.default_rng(7)
    nsam, nb = 64, 49_056 + 3
    g, ps, buf, ppar = _inputs(nsam, 2, rng)
    ctx = api.Context(0)
    ps = torch.from_numpy(ps).cuda()
    one = ctx.ctfapply(nsam, torch.from_numpy(buf.copy()).cuda(), torch.from_numpy(ppar).cuda(), ps,
                       g)
    pick = torch.arange(nb, device="cuda") % 2
    img = torch.from_numpy(buf).cuda()[pick].contiguous()
    par = torch.from_numpy(ppar).cuda()[pick].contiguous()
    many = ctx.ctfapply(nsam, img, par, ps, g)
    for x, y in zip(one, many):
        for b in (0, 1, nb // 2, 49_055, 49_056, 49_057, nb - 1):
            assert torch.equal(torch.view_as_real(x[b % 2]), torch.view_as_real(y[b]))
    ctx.close()
