"""What this framework's speed is measured on: the calls of a refinement cycle.

Each case is one public entry point at the sizes a job gives it:

  score      CC3M of (particle, orientation, shift) items: one round of PREFINE on a
             few particles (the smallest call), the rescoring of a search's
             candidates, and late cycles whose band is wide
  prep       LMAIN's r2c and CTFAPPLY for a batch of raw images
  search     the exhaustive orientation search, BF16 and FP32
  lists      the search over the learned proposal's candidate lists, with rescoring
  local      mode 1's grid of orientations and shifts around the known parameters
  refine     PREFINE (Powell's VA04A, lock-stepped) of a batch
  insert     A3D3's insertion into the two half-maps
  train      forward and backward of the proposal network in mixed precision

Particles are Gaussian-blob phantoms seen through a 300 kV CTF with white noise.
They are made with plain torch in 64 bits, so the inputs depend on the seed alone.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from frealign_amd import api, proposal, search, synth

DEV = "cuda"
PSIZE = 1.0
_CTX = None

# box sizes of the repository's tests and benchmark, and sizes between them (2^a 3^b 5^c, even)
BOXES = (64, 72, 80, 96, 100, 120, 128, 144, 160, 180, 192, 200, 216, 240, 250, 256, 288, 300,
         320, 360, 384)


def _ctx():
    """The one library context a program keeps."""
    global _CTX
    if _CTX is None:
        _CTX = api.Context(0)
    return _CTX


# ------------------------------------------------------------------- cases
def listed():
    return [
        # one objective evaluation of PREFINE for a handful of small particles: latency
        dict(name="score-small", op="score", nsam=64, maxr2=16, npart=8, ncand=1, mag=False),
        # the top-32 candidates of a search rescored (the benchmark's step, 8 A band)
        dict(name="score-rescore", op="score", nsam=256, maxr2=32, npart=256, ncand=32, mag=False),
        # a late cycle: large box, 4 A band
        dict(name="score-wide", op="score", nsam=320, maxr2=80, npart=128, ncand=4, mag=False),
        # preparation of a batch of raw images
        dict(name="prep", op="prep", nsam=256, nb=512),
        # exhaustive search at 5 degrees, D7: BF16, and the plain FP32 search beside it
        dict(name="search-bf16", op="search", nsam=256, maxr2=32, sym="D7", dang=5.0, np=128,
             bf16=True),
        dict(name="search-fp32", op="search", nsam=256, maxr2=32, sym="D7", dang=5.0, np=64,
             bf16=False),
        # the learned search: lists of the 8 proposed classes, then the FP32 rescoring
        dict(name="search-lists", op="lists", nsam=256, maxr2=32, sym="D7", dang=5.0, np=256),
        # mode 1: +-6 degrees at 1 degree, 9 x 9 shifts
        dict(name="local", op="local", nsam=128, maxr2=25, nang=6, nsh=4, np=24),
        # PREFINE of a batch's winners
        dict(name="refine", op="refine", nsam=256, maxr2=32, np=256),
        # insertion: a symmetric particle at a large box, and an asymmetric one at an odd size
        dict(name="insert-d7", op="insert", nsam=256, sym="D7", nb=64),
        dict(name="insert-c1", op="insert", nsam=150, sym="C1", nb=300),
        # one gradient of the proposal network
        dict(name="train", op="train", size=64, nconv=4, sym="D7", class_deg=15.0, batch=256),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _band(rng, n, top=0.45):
    """A resolution limit between 10 A and 2.2 A at 1 A per pixel."""
    return max(8, min(int(n * rng.uniform(0.1, top)), n // 2 - 2))


def draw(rng):
    op = rng.choice(["score", "score", "score", "prep", "prep", "search", "search", "lists",
                     "local", "refine", "insert", "insert", "train"])
    if op == "score":
        n = rng.choice(BOXES)
        items = _log(rng, 1, max(2, min(8192, 512 * 65536 // (n * n))))
        ncand = rng.choice([1, 1, 4, 16, 32])
        maxr2 = min(32, _band(rng, n)) if rng.random() < 0.5 else _band(rng, n)
        return dict(op=op, nsam=n, maxr2=maxr2, npart=max(1, items // ncand), ncand=ncand,
                    mag=rng.random() < 0.15)
    if op == "prep":
        n = rng.choice(BOXES)
        return dict(op=op, nsam=n, nb=_log(rng, 1, max(2, min(1024, 512 * 65536 // (n * n)))))
    if op == "search":
        n = rng.choice([96, 128, 160, 180, 192, 216, 256])
        return dict(op=op, nsam=n, maxr2=rng.randint(14, 40), sym=rng.choice(["D7", "D5", "O"]),
                    dang=rng.choice([4.0, 5.0, 6.0]), np=_log(rng, 2, 64), bf16=rng.random() < 0.6)
    if op == "lists":
        return dict(op=op, nsam=rng.choice([128, 160, 192, 256]), maxr2=rng.randint(16, 32),
                    sym=rng.choice(["D7", "D5"]), dang=rng.choice([4.0, 5.0, 6.0]),
                    np=_log(rng, 8, 256))
    if op == "local":
        return dict(op=op, nsam=rng.choice([64, 96, 128, 160, 192, 224, 256]),
                    maxr2=rng.randint(14, 31), nang=rng.randint(2, 6), nsh=rng.randint(1, 5),
                    np=_log(rng, 2, 24))
    if op == "refine":
        n = rng.choice(BOXES[2:17])
        return dict(op=op, nsam=n, maxr2=min(32, _band(rng, n)), np=_log(rng, 16, 256))
    if op == "insert":
        n = rng.choice(BOXES)
        sym = rng.choice(["C1", "C1", "C4", "D2", "D7", "O"])
        copies = {"C1": 1, "C4": 4, "D2": 4, "D7": 14, "O": 24}[sym]
        most = max(2, min(512, 700 * 65536 // (n * n * copies)))
        return dict(op=op, nsam=n, sym=sym, nb=_log(rng, 1, most))
    return dict(op=op, size=rng.choice([32, 64, 64, 128]), nconv=rng.randint(3, 4),
                sym=rng.choice(["D7", "D4"]), class_deg=rng.choice([12.0, 15.0, 18.0]),
                batch=_log(rng, 24, 256))


# ------------------------------------------------------------------ inputs
def _rng(case, seed, salt):
    g = torch.Generator(device=DEV)
    g.manual_seed((int(seed) * 1_000_003 + salt) % (1 << 62))
    return g


def _nrng(seed, salt):
    return np.random.default_rng([int(seed) % (1 << 32), salt])


def _freq(n):
    """Column and (wrapped) row indices of the half-plane."""
    jc = n // 2 + 1
    col = torch.arange(jc, device=DEV)
    row = torch.arange(n, device=DEV)
    return col, torch.where(row >= jc, row - n, row)


def _point_group(name):
    return api.point_group(name[0], int(name[1:]) if len(name) > 1 else 1)


def _volume(n, sym, seed):
    """The half-volume of a phantom of Gaussian blobs, with the point group's copies."""
    r = _nrng(seed, 1)
    mats = synth.symmetry_matrices(sym)
    nblob = 40
    u = r.standard_normal((nblob, 3))
    u *= (0.4 * n * r.uniform(0, 1, nblob) ** (1 / 3) / np.linalg.norm(u, axis=1))[:, None]
    cen = torch.from_numpy(np.concatenate([u @ m.T for m in mats])).to(DEV)
    sig = torch.from_numpy(np.tile(r.uniform(0.008, 0.02, nblob) * n, len(mats))).to(DEV)
    amp = torch.from_numpy(np.tile(r.uniform(0.5, 1.0, nblob), len(mats))).to(DEV)
    x = torch.arange(n, device=DEV, dtype=torch.float64) - n // 2
    e = torch.exp(-((x[None, None] - cen[:, :, None]) ** 2) / (2 * sig[:, None, None] ** 2))
    ex, ey, ez = e[:, 0], e[:, 1], e[:, 2] * amp[:, None]
    vol = torch.zeros((n * n, n), device=DEV, dtype=torch.float64)
    for b in range(0, len(cen), 64):
        zy = (ez[b:b + 64, :, None] * ey[b:b + 64, None, :]).reshape(-1, n * n)
        vol += zy.T @ ex[b:b + 64]
    return synth.half_volume(vol.reshape(n, n, n))


def _section(a3df, dm, ci, cj):
    """AINTERPO3DS in 64 bits at the points (ci, cj) of the planes dm (k, 9): the
    coordinates as the reference forms them in FP32, the weights and sums in 64 bits."""
    n = a3df.shape[0]
    jc = n // 2 + 1
    flat = a3df.reshape(-1)
    fi, fj = ci.float()[None], cj.float()[None]
    x, y, z = (dm[:, k:k + 1] * fi + dm[:, 3 + k:4 + k] * fj for k in range(3))
    neg = x < 0
    x, y, z = (torch.where(neg, -v, v).double() for v in (x, y, z))
    out = 0
    lx, my, nz = (torch.floor(v).long() for v in (x, y, z))
    for bz in (0, 1):
        n1 = (nz + bz).clamp(-jc + 1, jc - 1)
        wz = 1 - (z - n1).abs()
        for by in (0, 1):
            m1 = (my + by).clamp(-jc + 1, jc - 1)
            wy = wz * (1 - (y - m1).abs())
            for bx in (0, 1):
                l1 = (lx + bx).clamp(0, jc - 1)
                w = wy * (1 - (x - l1).abs())
                out = out + flat[l1 + jc * ((m1 % n) + n * (n1 % n))].to(torch.complex128) * w
    return torch.where(neg, out.conj(), out)


def _chi(n, df1, df2, ang):
    """The phase of ctf.f on the half-plane, 64 bits, for k particles."""
    o = synth.Optics(psize=PSIZE)
    g = o.gpar(n, 0.45 * n)
    col, row = _freq(n)
    L, M = col.double()[None, :], row.double()[:, None]
    angle = torch.sqrt(L * L + M * M) * float(g[4])
    c1 = 2 * math.pi * angle * angle / (2.0 * float(g[1]))
    c2 = c1 * float(g[0]) * angle * angle / 2.0
    ccos = torch.cos(2.0 * (torch.atan2(M, L)[None] - ang[:, None, None]))
    d1, d2 = df1[:, None, None], df2[:, None, None]
    return c1[None] * (-0.5 * (d1 + d2 + ccos * (d1 - d2))) + c2[None]


def _ctf(n, df1, df2, ang):
    """CTFR = CTFL without beam tilt, (k, n, jc) complex128."""
    g = synth.Optics(psize=PSIZE).gpar(n, 0.45 * n)
    w1, w2 = float(g[2]), abs(float(g[3]))
    chi = _chi(n, df1, df2, ang)
    s, c = torch.sin(chi), torch.cos(chi)
    out = torch.complex(w1 * s - w2 * c, -w1 * c - w2 * s)
    out[:, 0, 0] = -w2
    return out


def _particles(n, count, a3df, seed, snr=0.05, euler=None):
    """Noisy particle spectra (count, n, jc) c64, their CTF tables (count, 2, n, jc),
    the true angles (count, 3), shifts (count, 2) and defocus records (count, 3)."""
    r = _nrng(seed, 2)
    jc = n // 2 + 1
    eul = synth.random_orientations(count, r) if euler is None else euler
    sh = (r.uniform(-3, 3, (count, 2)) / n * 2 * math.pi).astype(np.float32)
    df = r.uniform(1.0e4, 3.0e4, count)
    ast = r.uniform(0, 1.0e3, count)
    rec = np.stack([df + ast / 2, df - ast / 2, r.uniform(-math.pi, math.pi, count)],
                   1).astype(np.float32)
    dm = torch.from_numpy(api.rotation(eul, amag=0.0)).to(DEV)
    col, row = _freq(n)
    L, M = col[None, :].expand(n, jc), row[:, None].expand(n, jc)
    inside = (L * L + M * M <= (n // 2 - 1) ** 2).reshape(-1)
    pts = torch.nonzero(inside)[:, 0]
    ci, cj = L.reshape(-1)[pts], M.reshape(-1)[pts]
    spec = torch.empty((count, n, jc), dtype=torch.complex64, device=DEV)
    ctff = torch.empty((count, 2, n, jc), dtype=torch.complex64, device=DEV)
    g = _rng(None, seed, 3)
    step = max(1, (1 << 22) // (n * jc))
    for b in range(0, count, step):
        e = min(count, b + step)
        t = [torch.from_numpy(rec[b:e, k]).to(DEV).double() for k in range(3)]
        c = _ctf(n, *t)
        sec = torch.zeros((e - b, n * jc), dtype=torch.complex128, device=DEV)
        sec[:, pts] = _section(a3df, dm[b:e], ci, cj)
        sec = sec.reshape(e - b, n, jc) * (2 * c.real)
        s = torch.from_numpy(sh[b:e]).to(DEV).double()
        ph = -(s[:, 0, None, None] * L + s[:, 1, None, None] * M)
        sec = sec * torch.polar(torch.ones_like(ph), ph)
        noise = torch.fft.rfft2(torch.randn((e - b, n, n), generator=g, device=DEV).double())
        std = torch.sqrt((sec.abs() ** 2).mean(dim=(1, 2), keepdim=True) / snr) / n
        x = sec + noise * std
        x = x / (x.abs() ** 2).mean(dim=(1, 2), keepdim=True).sqrt()
        spec[b:e] = x.to(torch.complex64)
        ctff[b:e, 0] = c.to(torch.complex64)
        ctff[b:e, 1] = ctff[b:e, 0]
    return spec, ctff, eul, sh, rec


def _ring(n):
    g = synth.Optics(psize=PSIZE).gpar(n, 0.45 * n)
    return np.array([g[7], g[8], g[5], g[6]], np.float32)


def _dev(a, dtype=None):
    return torch.from_numpy(np.ascontiguousarray(a, dtype)).to(DEV)


def prepare(case, seed):
    ctx, op = _ctx(), case["op"]
    s = dict(case, ctx=ctx)
    if op == "train":
        sym = _point_group(case["sym"])
        mats = synth.symmetry_matrices(sym)
        cls = proposal.OrientationClasses(case["class_deg"], case["sym"][0], int(case["sym"][1:]),
                                          mats)
        r = _nrng(seed, 4)
        shape = (case["size"], 64, case["nconv"], cls.n)
        count = api.cnn_param_count(*shape)
        s["master"], s["wq"], s["grad"] = (torch.zeros(count, device=DEV) for _ in range(3))
        ctx.cnn_init(shape, int(seed) + 1, s["master"], s["wq"])
        g = _rng(case, seed, 5)
        # each class has an image of its own under the noise, normalised as the crop is
        base = torch.randn((cls.n, case["size"], case["size"]), generator=g, device=DEV)
        lab = r.integers(0, cls.n, case["batch"])
        s["label"] = _dev(lab, np.int32)
        img = 0.3 * base[s["label"].long()] + torch.randn(
            (case["batch"], case["size"], case["size"]), generator=g, device=DEV)
        m = img.mean(dim=(1, 2), keepdim=True)
        s["img"] = ((img - m) / img.std(dim=(1, 2), keepdim=True)).contiguous()
        s["shape"] = shape
        return s
    n = case["nsam"]
    sym = _point_group(case.get("sym", "C1"))
    a3df = _volume(n, sym, seed)
    s.update(a3df=a3df, ring=_ring(n), fsct=_dev(synth.default_fsct(n, PSIZE)), maxr1=2)
    if op == "prep":
        spec, ctff, eul, sh, rec = _particles(n, case["nb"], a3df, seed)
        col, row = _freq(n)
        sgn = 1 - 2 * ((col[None, :] + row[:, None]) % 2)
        img = torch.zeros((case["nb"], n, n + 2), device=DEV)
        img[:, :, :n] = torch.fft.irfft2(spec * sgn, s=(n, n)) * n
        p = np.zeros((case["nb"], 8), np.float32)
        p[:, 0:2], p[:, 2:5], p[:, 5] = 0.5 * sh, rec, 1.0
        o = synth.Optics(psize=PSIZE)
        s.update(images=img, ppar=_dev(p), pssnr=_dev(synth.default_pssnr(n, 0.45 * n)),
                 gpar=o.gpar(n, 0.45 * n))
        return s
    count = case["npart"] if op == "score" else case["nb"] if op == "insert" else case["np"]
    spec, ctff, eul, sh, rec = _particles(n, count, a3df, seed, snr=0.1 if op == "local" else 0.05)
    s.update(spec=spec, ctff=ctff)
    r = _nrng(seed, 6)
    if op == "score":
        k = case["ncand"]
        e = np.repeat(eul, k, 0) + r.normal(0, 0.06, (count * k, 3))
        am = r.uniform(0.97, 1.03, count * k) if case["mag"] else np.ones(count * k)
        dm = api.rotation(e.astype(np.float32), amag=1.0) / am[:, None].astype(np.float32)
        d = np.repeat(sh, k, 0) + r.normal(0, 2.0 / n, (count * k, 2))
        s.update(pidx=_dev(np.repeat(np.arange(count), k), np.int32), dm=_dev(dm, np.float32),
                 shift=_dev(d, np.float32), amag=_dev(am, np.float32))
    elif op in ("search", "lists"):
        bf16 = op == "lists" or case["bf16"]
        gs = search.GlobalSearch(ctx, a3df, dang=case["dang"], asym=case["sym"][0],
                                 nasym=int(case["sym"][1:] or 1), maxr1=2, maxr2=case["maxr2"],
                                 rbfact=0.0, dtype=torch.bfloat16 if bf16 else torch.float32,
                                 iran=-7 - int(seed) % 1000)
        s["gs"] = gs
        if op == "lists":
            # the 8 classes nearest to the truth stand for the network's answer, and
            # one particle in 64 falls back to the whole bank
            mats = synth.symmetry_matrices(sym)
            lp = proposal.LearnedProposal(ctx, gs, mats, case["sym"][0], int(case["sym"][1:]))
            t = _dev(api.rotation(eul, amag=0.0)).reshape(-1, 3, 3).double()
            c = _dev(lp.classes.dm).reshape(-1, 3, 3).double()
            tr = torch.stack([((t @ _dev(m.T).double()).reshape(count, 9)
                               @ c.reshape(-1, 9).T) for m in mats]).amax(0)
            s["lp"] = lp
            s["top"] = torch.topk(tr, 8, dim=1).indices.to(torch.int32).contiguous()
            conf = r.uniform(0.35, 0.9, count)
            conf[r.uniform(0, 1, count) < 1 / 64] = 0.2
            prob = np.concatenate([conf[:, None], np.repeat((1 - conf)[:, None] / 8, 7, 1)], 1)
            s["prob"] = _dev(prob, np.float32)
    elif op == "local":
        par = np.concatenate([eul + r.normal(0, 0.04, eul.shape),
                              sh + r.normal(0, 3.0 / n, sh.shape)], 1)
        s.update(par=par.astype(np.float32), dang=float(np.float32(math.pi / 180)),
                 dsh=float(np.float32(2 * math.pi / n)))
    elif op == "refine":
        par = np.zeros((count, 6), np.float32)
        par[:, :3] = eul + r.normal(0, 0.03, eul.shape)
        par[:, 3:5] = sh + r.normal(0, 1.5 / n, sh.shape)
        prior = np.zeros((count, 5), np.float32)
        prior[:, 2:4], prior[:, 4] = 0.05, 0.01
        s.update(par=par, prior=prior, pidx=np.arange(count, dtype=np.int32),
                 amag=np.ones(count, np.float32), mask=np.ones(5, np.int32))
    elif op == "insert":
        rb = np.zeros((count, 10), np.float32)
        rb[:, 0:3], rb[:, 3:5], rb[:, 5:8], rb[:, 8:10] = eul, sh, 1.0, 0.5
        rb[:, 6] = r.uniform(0.5, 1.0, count)
        s.update(recb=rb, half=(np.arange(count) % 2).astype(np.int32), sym=sym,
                 vols=api.HalfMaps.zeros(n))
    return s


# --------------------------------------------------------------------- run
def run(s):
    ctx, op = s["ctx"], s["op"]
    if op == "train":
        loss = ctx.cnn_gradients(s["shape"], s["wq"], s["img"], s["label"], s["grad"], bf16=True)
        return {"loss": loss, "grad": s["grad"]}
    n = s["nsam"]
    if op == "prep":  # the transform is in place: a batch comes in a buffer of its own
        ctff, outc, datc = ctx.ctfapply(n, s["images"].clone(), s["ppar"], s["pssnr"], s["gpar"])
        return {"ctff": ctff, "outc": outc, "datc": datc}
    if op == "score":
        return ctx.cc3m(n, s["a3df"], s["spec"], s["ctff"], s["pidx"], s["dm"], s["shift"],
                        s["amag"], s["maxr1"], s["maxr2"], 0.0, s["fsct"], s["ring"])
    if op == "search":
        o, r, sc = s["gs"].candidates(s["spec"], s["ctff"], 32)
        return {"view": o, "row": r, "score": sc}
    if op == "lists":
        gs, lp = s["gs"], s["lp"]
        loff, grp, cand, info = ctx.build_lists(s["top"], s["prob"], lp.cfg.threshold,
                                                lp.cell_off_dev, lp.cells_dev, lp.cfg.group,
                                                gs.norient, gs.group, lp.maxlen)
        o, r, sc = ctx.search_ragged(n, gs.maxr1, gs.maxr2, gs.rbfact, gs.search_bank, s["spec"],
                                     s["ctff"], loff, grp, cand, 32, info=info)
        fs, best = ctx.rescore(n, s["a3df"], s["spec"], s["ctff"], o, r, gs.dm, gs.nsamr, gs.maxr1,
                               gs.maxr2, gs.rbfact, s["fsct"], s["ring"])
        return {"view": o, "row": r, "score": sc, "cc3m": fs, "best": best}
    if op == "local":
        p, sc, code = ctx.local_search(n, s["a3df"], s["spec"], s["ctff"], s["par"],
                                       nang=s["nang"], dang=s["dang"], nsh=s["nsh"], dsh=s["dsh"],
                                       maxr1=s["maxr1"], maxr2=s["maxr2"], rbfact=0.0,
                                       fsct=s["fsct"], ring=s["ring"], all_scores=True)
        return {"par": p, "score": sc, "shift": code}
    if op == "refine":
        p, nev = ctx.refine(n, s["a3df"], s["spec"], s["ctff"], s["pidx"], s["amag"], s["par"],
                            s["mask"], s["maxr1"], s["maxr2"], 0.0, s["fsct"], s["ring"],
                            s["prior"])
        return {"par": p}  # how many evaluations it took is the path's own affair
    v = s["vols"]  # a cycle's maps, from zero, so that a pass can be made again
    for t in (*v.num, *v.ctf2, v.nksum, v.ttd):
        t.zero_()
    ctx.insert(n, s["spec"], s["ctff"], s["recb"], s["half"], s["sym"], 5.0, 40.0, PSIZE, v)
    return {"num": list(v.num), "ctf2": list(v.ctf2), "count": v.nksum, "ttd": v.ttd}


# ------------------------------------------------------------ work, tolerance
def _score_work(items, npart, n, maxr2, shifts=1):
    """Per item: eight corners of each band point, the CTF, a transform pair on the
    smallest grid that holds the masked band (twice its width), the shell sums."""
    pts = math.pi * maxr2 * maxr2 / 2
    m = min(n, 4 * maxr2)
    flops = items * (pts * (48 + 8 + 14 * shifts) + 2 * 5 * m * m * math.log2(m * m) / 2)
    return {"bytes": npart * pts * 24 + items * 56 + min(n, 2 * maxr2) ** 3 * 4, "flops": flops}


def work(case):
    op = case["op"]
    if op == "train":
        ch, ci, h, f = 64, 1, case["size"], 0.0
        for _ in range(case["nconv"]):
            h //= 2
            f += 2 * ch * ci * 9 * h * h * (3 if ci > 1 else 2)
            ci = ch
        classes = 100
        f += 6 * ch * h * h * classes
        par = ch * 9 + (case["nconv"] - 1) * ch * ch * 9 + ch * h * h * classes
        return {"bytes": case["batch"] * case["size"] ** 2 * 4 + par * 8, "flops": case["batch"] * f}
    n = case["nsam"]
    plane = n * (n // 2 + 1)
    if op == "prep":
        return {"bytes": case["nb"] * plane * (8 + 16 + 8 + 8),
                "flops": case["nb"] * (3 * 2.5 * n * n * math.log2(n * n) + 60.0 * plane)}
    if op == "score":
        return _score_work(case["npart"] * case["ncand"], case["npart"], n, case["maxr2"])
    pts = math.pi * case.get("maxr2", 0) ** 2 / 2
    if op in ("search", "lists"):
        # per pair: the product and its norm, and the 15 x 15 shifts one axis at a time
        grid = case["maxr2"] * 2 * case["maxr2"]
        pairs = case["np"] * (1000 if op == "lists" else 46800 * (5.0 / case["dang"]) ** 3)
        f = pairs * (pts * 12 + 8 * 15 * grid + 4 * 225 * case["maxr2"])
        w = {"bytes": case["np"] * pts * 24 + 46800 * (5.0 / case["dang"]) ** 3 * pts *
             (4 if op == "lists" or case["bf16"] else 8), "flops": f}
        if op == "lists":
            more = _score_work(case["np"] * 32, case["np"], n, case["maxr2"])
            w = {k: w[k] + more[k] for k in w}
        return w
    if op == "local":
        items = case["np"] * (2 * case["nang"] + 1) ** 3
        return _score_work(items, case["np"], n, case["maxr2"], (2 * case["nsh"] + 1) ** 2)
    if op == "refine":
        return _score_work(case["np"] * 60, case["np"], n, case["maxr2"])
    copies = {"C1": 1, "C4": 4, "D2": 4, "D7": 14, "O": 24}[case["sym"]]
    pts = math.pi * (n // 2) ** 2 / 2
    return {"bytes": case["nb"] * plane * 24 + 2 * 12 * n * plane,
            "flops": case["nb"] * (pts * 40 + copies * pts * (15 + 8 * 9))}


def tolerance(case):
    op = case["op"]
    if op == "train":  # operands round to BF16: a rounding apart, one falls on the next value
        return {"rel": 1e-2, "max": 0.3}
    if op == "prep":  # the CTF's phase is hundreds of radians in FP32: 2.4e-5 off exact()
        return {"rel": 1e-4, "max": 5e-3}
    if op == "refine":  # a rounding apart, VA04A stops elsewhere on a flat top
        return {"rel": 5e-3, "max": 0.2}
    if op == "local":  # two grid points that tie to a rounding may change places
        return {"rel": 3e-3, "max": 0.1, "differ": 0.01}
    if op == "lists" or (op == "search" and case["bf16"]):  # ties in the list of the best
        return {"rel": 1e-2, "max": 0.1, "differ": 0.01}
    if op == "search":
        return {"rel": 2e-5, "max": 1e-3, "differ": 0.01}
    if op == "insert":
        return {"rel": 2e-6, "max": 1e-4}
    return {"rel": 2e-5, "max": 1e-3}


# ------------------------------------------------------------------- exact
def _annulus(n, lo2, hi2):
    """Half-plane points with lo2 <= r^2 < hi2 (r < n/2), I >= 0 and both signs of J."""
    col, row = _freq(n)
    L, M = col[None, :].expand(n, len(col)), row[:, None].expand(n, len(col))
    r2 = L * L + M * M
    pts = torch.nonzero(((r2 >= lo2) & (r2 < hi2)).reshape(-1))[:, 0]
    return pts, L.reshape(-1)[pts], M.reshape(-1)[pts]


def _masked_band(n, a, pts, ring, am):
    """The band values `a` (k, points) through c2r, MASKCOS2 about the origin and r2c."""
    k = a.shape[0]
    f = torch.zeros((k, n * (n // 2 + 1)), dtype=torch.complex128, device=DEV)
    f[:, pts] = a / (n * n)
    x = torch.fft.irfft2(f.reshape(k, n, -1), s=(n, n), norm="forward")
    d = torch.arange(n, device=DEV)
    d = torch.where(d < n // 2, d, d - n).double()
    r2 = d[:, None] ** 2 + d[None, :] ** 2
    ri2, ri3, rih, halfw = (float(v) for v in ring)
    am = am.double()[:, None, None]
    inner, outer = r2[None] > ri2 / am / am, r2[None] > ri3 / am / am
    edge = (1 + torch.cos(math.pi * (torch.sqrt(r2)[None] - rih / am) / halfw)) / 2
    w = torch.where(outer, torch.zeros_like(edge), torch.where(inner, edge, torch.ones_like(edge)))
    rim = (inner & ~outer).double()
    mean = (x * rim).sum((1, 2)) / rim.sum((1, 2)).clamp_min(1)
    x = x * w + (1 - w) * mean[:, None, None]
    return torch.fft.rfft2(x).reshape(k, -1)[:, pts]


def _shells(ci, cj):
    return (torch.sqrt((ci * ci + cj * cj).float()) + 0.5).long()


def _exact_score(s, a3df, spec, ctff, pidx, dm, am, windows):
    """CC3M of every item at the shifts `windows` (items, s, 2), 64 bits."""
    n = a3df.shape[0]
    pts, ci, cj = _annulus(n, s["maxr1"] ** 2, s["maxr2"] ** 2)
    sh = _shells(ci, cj)
    order = torch.argsort(sh, stable=True)
    pts, ci, cj, sh = pts[order], ci[order], cj[order], sh[order]
    cnt = torch.bincount(sh, minlength=n // 2)
    off = [0] + torch.cumsum(cnt, 0).tolist()
    fsct = s["fsct"]
    out = torch.empty(windows.shape[:2], dtype=torch.float64, device=DEV)
    step = max(1, (1 << 24) // (n * n))
    for b in range(0, len(pidx), step):
        p = pidx[b:b + step].long()
        c = (ctff[p, 0].reshape(len(p), -1)[:, pts].to(torch.complex128)
             + ctff[p, 1].reshape(len(p), -1)[:, pts].to(torch.complex128).conj())
        a = _section(a3df, dm[b:b + step], ci, cj) * c
        a = _masked_band(n, a, pts, s["ring"], am[b:b + step])
        x = spec[p].reshape(len(p), -1)[:, pts].to(torch.complex128)
        prod = x * a.conj()
        w = windows[b:b + step].double()
        num = torch.zeros(w.shape[:2], dtype=torch.float64, device=DEV)
        s1, s2 = 0.0, torch.zeros(len(p), dtype=torch.float64, device=DEV)
        for k in range(1, n // 2):
            if off[k + 1] == off[k]:
                continue
            r = slice(off[k], off[k + 1])
            ph = w[:, :, :1] * ci[r].double() + w[:, :, 1:] * cj[r].double()
            q = (prod[:, None, r].real * torch.cos(ph) - prod[:, None, r].imag * torch.sin(ph)).sum(2)
            q = q / torch.sqrt((a[:, r].abs() ** 2).sum(1))[:, None]
            num += q.abs() if float(fsct[k]) < 0.95 else q
            s2 += (x[:, r].abs() ** 2).sum(1)
            s1 += 1
        out[b:b + step] = num / torch.sqrt(s1 * s2)[:, None]
    return out


def _exact_prep(s):
    n, nb = s["nsam"], s["nb"]
    jc = n // 2 + 1
    col, row = _freq(n)
    L, M = col[None, :].expand(n, jc), row[:, None].expand(n, jc)
    sgn = 1 - 2 * ((L + M) % 2)
    r2 = L * L + M * M
    g, pp, ssnr = s["gpar"], s["ppar"].double(), s["pssnr"].double()
    rih, halfw, ri2, ri3 = (float(v) for v in g[5:9])
    d = torch.arange(n, device=DEV, dtype=torch.float64) - n // 2
    c2 = d[:, None] ** 2 + d[None, :] ** 2
    inner, outer = c2 > ri2, c2 > ri3
    w = torch.where(outer, torch.zeros_like(c2), torch.where(
        inner, (1 + torch.cos(math.pi * (torch.sqrt(c2) - rih) / halfw)) / 2, torch.ones_like(c2)))
    rim = (inner & ~outer).double()
    # PWEIGHT's shells: J = -N/2 and +N/2 both address the Nyquist row, and the shell
    # beyond the last shares the place of the first one's count
    mult = torch.where(M == n // 2, 2.0, 1.0).double()
    band = r2 < jc * jc
    bins = torch.where(band, (torch.sqrt(r2.float()) + 0.5).long() + 1, 0)
    ctff, outc, datc = [], [], []
    for b in range(0, nb, 64):
        p = pp[b:b + 64]
        spec = torch.fft.rfft2(s["images"][b:b + 64, :, :n].double())
        c = _ctf(n, p[:, 2], p[:, 3], p[:, 4])
        ph = p[:, 0, None, None] * L + p[:, 1, None, None] * M
        v = spec * torch.polar(torch.ones_like(ph), ph)
        x = torch.fft.irfft2(v, s=(n, n))
        mean = (x * rim).sum((1, 2)) / rim.sum()
        o = torch.fft.rfft2(x * w + (1 - w) * mean[:, None, None]) * sgn
        power = torch.zeros((len(p), 2 * jc + 3), dtype=torch.float64, device=DEV)
        flat = bins.reshape(1, -1).expand(len(p), -1)
        power.scatter_add_(1, flat, ((o.abs() ** 2) * mult * band).reshape(len(p), -1))
        power.scatter_add_(1, torch.where(flat > 0, flat + jc, 0),
                           (mult * band).reshape(1, -1).expand(len(p), -1).contiguous())
        buf = power.clone()
        for i in range(1, jc + 1):
            den = buf[:, i + jc]
            buf[:, i] = torch.where(den != 0, torch.sqrt(buf[:, i] / den), buf[:, i])
            buf[:, i] = torch.where(buf[:, i] == 0, torch.ones_like(den), buf[:, i])
        snr = ssnr[(bins - 1).clamp_min(0)][None] * (2 * c.real) ** 2
        wgt = snr / (snr + 1) / buf[:, bins]
        wgt = torch.where(M == n // 2, wgt * wgt, wgt) * band
        ctff.append(torch.stack([c, c], 1))
        outc.append(torch.where(band, o * wgt, torch.zeros_like(o)))
        datc.append(v * sgn)
    return {"ctff": torch.cat(ctff), "outc": torch.cat(outc), "datc": torch.cat(datc)}


def _exact_search(s, rows=None):
    """The 32 best group scores of every particle, 64 bits.  rows: per particle the
    bank rows it lists and their group length (None: the whole bank by views)."""
    gs, n, npart = s["gs"], s["nsam"], s["np"]
    pts, ci, cj = _annulus(n, s["maxr1"] ** 2, s["maxr2"] ** 2)
    x = s["spec"].reshape(npart, -1).to(torch.complex128)
    c = (s["ctff"][:, 0].to(torch.complex128)
         + s["ctff"][:, 1].to(torch.complex128).conj()).reshape(npart, -1)[:, pts]
    sh = torch.arange(-7, 8, device=DEV).double() * (2 * math.pi / gs.nsamr)
    ph = (ci[:, None, None] * sh[None, :, None] + cj[:, None, None] * sh[None, None, :])
    ph = torch.polar(torch.ones_like(ph), ph).reshape(len(pts), 225)
    a = torch.where(ci > 0, 2.0, 1.0) * x[:, pts] * c.conj()
    a = (a[:, :, None] * ph[None]).transpose(1, 2).reshape(npart * 225, -1)
    low, li, lj = _annulus(n, 1, s["maxr2"] ** 2)
    both = torch.where((li == 0) & (lj.abs() == n // 2), 2.0, 1.0)
    s2 = ((x[:, low].abs() ** 2) * both).sum(1)
    score = torch.empty((npart, gs.norient), dtype=torch.float64, device=DEV)
    step = max(64, (1 << 26) // (npart * 225))
    for b in range(0, gs.norient, step):
        t = _section(s["a3df"], gs.dm[b:b + step], ci, cj)
        cc = (a.real @ t.real.T + a.imag @ t.imag.T).reshape(npart, 15, 15, -1)
        inner = cc[:, 1:14, 1:14].reshape(npart, 169, -1)
        at = inner.argmax(1)
        box = sum(torch.gather(cc[:, dx:dx + 13, dy:dy + 13].reshape(npart, 169, -1), 1,
                               at[:, None])[:, 0] for dx in range(3) for dy in range(3))
        nrm = (c.abs() ** 2) @ (t.abs() ** 2).T
        score[:, b:b + step] = box / torch.sqrt(nrm) / torch.sqrt(s2)[:, None] / 9
    if rows is None:
        best = score.reshape(npart, -1, gs.group).amax(2)
        return torch.topk(best, 32, dim=1).values
    out = torch.empty((npart, 32), dtype=torch.float64, device=DEV)
    for p, (r, g) in enumerate(rows):
        v = torch.where(r >= 0, score[p][r.clamp_min(0)], -math.inf)
        out[p] = torch.topk(v.reshape(-1, g).amax(1), 32).values
    return out


def _exact_insert(s):
    n, nb = s["nsam"], s["nb"]
    jc, h = n // 2 + 1, n // 2
    nsym, symop, jsym, _ = s["sym"]
    num = [torch.zeros((n * n * jc, 2), dtype=torch.float64, device=DEV) for _ in range(2)]
    ctf2 = [torch.zeros(n * n * jc, dtype=torch.float64, device=DEV) for _ in range(2)]
    ttd = [0.0, 0.0]
    col = torch.arange(-h, h + 1, device=DEV)
    I, J = (v.reshape(-1) for v in torch.meshgrid(col, col, indexing="ij"))
    rec = s["recb"]
    rr = int(np.float32(n) * rec[0, 9])
    keep = I * I + J * J <= rr * rr
    I, J = I[keep], J[keep]
    g2 = (I * I + J * J).double()
    at = torch.where(I >= 0, I + jc * (J % n), -I + jc * ((-J) % n))
    for p in range(nb):
        r = rec[p].astype(np.float64)
        occ = r[6] / r[7]
        tmp = min((r[8] / 0.05 - 40.0 / 5.0) / (PSIZE * PSIZE), 2.0)
        wgt = torch.exp(2 * tmp / (h * h) * g2) * occ
        v = s["spec"][p].reshape(-1)[at].to(torch.complex128)
        v = torch.where(I >= 0, v, v.conj())
        ph = float(rec[p, 3]) * I.double() + float(rec[p, 4]) * J.double()
        c = (s["ctff"][p, 0].reshape(-1)[at].to(torch.complex128)
             + s["ctff"][p, 1].reshape(-1)[at].to(torch.complex128).conj())
        v = v * torch.polar(torch.ones_like(ph), ph) * c * wgt
        t = 0.25 * c.abs() ** 2 * wgt
        first = api.rotation(rec[p:p + 1, 0:3], amag=float(rec[p, 5]))[0]
        half = int(s["half"][p])
        for copy in np.ndindex(*[int(j) for j in jsym[:nsym]]):
            dm = first.copy()
            for k, power in enumerate(copy):
                for _ in range(power):
                    op = symop[9 * k:9 * k + 9].reshape(3, 3).astype(np.float32)
                    new = np.empty(9, np.float32)  # FP32, in the order of matmul_t.f
                    for q in range(3):
                        for u in range(3):
                            x = np.float32(dm[3 * q] * op[u, 0])
                            x = np.float32(x + np.float32(dm[3 * q + 1] * op[u, 1]))
                            new[3 * q + u] = np.float32(x + np.float32(dm[3 * q + 2] * op[u, 2]))
                    dm = new
            x3 = [(float(dm[k]) * I.float() + float(dm[3 + k]) * J.float()).double()
                  for k in range(3)]
            base = [torch.floor(q).long() for q in x3]
            for bx in (0, 1):
                l1 = base[0] + bx
                okx = (l1 >= 0) & (l1 <= h)
                wx = 1 - (x3[0] - l1).abs()
                for by in (0, 1):
                    m1 = base[1] + by
                    oky = okx & (m1.abs() <= h)
                    wy = wx * (1 - (x3[1] - m1).abs())
                    for bz in (0, 1):
                        n1 = base[2] + bz
                        ok = oky & (n1.abs() <= h)
                        w = torch.where(ok, wy * (1 - (x3[2] - n1).abs()), 0.0)
                        idx = torch.where(ok, l1 + jc * ((m1 % n) + n * (n1 % n)), 0)
                        num[half].index_add_(0, idx, torch.view_as_real(v * w))
                        ctf2[half].index_add_(0, idx, t * w)
                        ttd[half] = ttd[half] + (t * w).sum()
    shape = (n, n, jc)
    return {"num": [torch.view_as_complex(q).reshape(shape) for q in num],
            "ctf2": [q.reshape(shape) for q in ctf2], "count": None,
            "ttd": torch.stack([torch.as_tensor(q, dtype=torch.float64, device=DEV) for q in ttd])}


def _exact_train(s):
    size, ch, nconv, classes = s["shape"]
    w = s["wq"].double().requires_grad_(True)
    x, at, ci = s["img"].double()[:, None], 0, 1
    for _ in range(nconv):
        k = w[at:at + ch * ci * 9].reshape(ch, ci * 9)
        at += ch * ci * 9
        cols = torch.nn.functional.unfold(x, 3, padding=1, stride=2)
        x = torch.relu(k @ cols + w[at:at + ch][:, None])
        at += ch
        size //= 2
        x, ci = x.reshape(-1, ch, size, size), ch
    f = ch * size * size
    logits = x.reshape(-1, f) @ w[at:at + classes * f].reshape(classes, f).T
    logits = logits + w[at + classes * f:at + classes * f + classes]
    loss = torch.logsumexp(logits, 1) - logits[torch.arange(len(logits)), s["label"].long()]
    loss.mean().backward()
    return {"loss": loss.detach(), "grad": w.grad}


def exact(case, seed):
    op = case["op"]
    if op == "refine":
        return None
    s = prepare(case, seed)
    if op == "train":
        return _exact_train(s)
    if op == "prep":
        return _exact_prep(s)
    if op == "score":
        return _exact_score(s, s["a3df"], s["spec"], s["ctff"], s["pidx"], s["dm"], s["amag"],
                            s["shift"][:, None])[:, 0]
    if op == "search":
        return {"view": None, "row": None, "score": _exact_search(s)}
    if op == "lists":
        gs, lp, rows = s["gs"], s["lp"], []
        whole = torch.arange(gs.norient, device=DEV)
        for p in range(s["np"]):
            if float(s["prob"][p, 0]) < lp.cfg.threshold:
                rows.append((whole, gs.group))
            else:
                r = np.concatenate([lp.cells[c] for c in s["top"][p].tolist()])
                rows.append((_dev(r, np.int64), lp.cfg.group))
        return {"view": None, "row": None, "score": _exact_search(s, rows), "cc3m": None,
                "best": None}
    if op == "local":
        k = np.arange(-s["nang"], s["nang"] + 1, dtype=np.float32) * np.float32(s["dang"])
        a, b, c = (v.reshape(-1) for v in np.meshgrid(k, k, k, indexing="ij"))
        q = np.arange(-s["nsh"], s["nsh"] + 1) * np.float32(s["dsh"])
        dx, dy = (v.reshape(-1) for v in np.meshgrid(q, q, indexing="ij"))
        best = []
        for p in range(s["np"]):
            e = np.stack([s["par"][p, 0] + a, s["par"][p, 1] + b, s["par"][p, 2] + c], 1)
            dm = _dev(api.rotation(e.astype(np.float32), amag=1.0))
            w = _dev(np.stack([s["par"][p, 3] + dx, s["par"][p, 4] + dy], 1))
            w = w[None].expand(len(a), -1, -1)
            pidx = torch.full((len(a),), p, device=DEV)
            sc = _exact_score(s, s["a3df"], s["spec"], s["ctff"], pidx, dm,
                              torch.ones(len(a), device=DEV), w)
            best.append(sc.amax(1))
        return {"par": None, "score": torch.stack(best), "shift": None}
    return _exact_insert(s)
