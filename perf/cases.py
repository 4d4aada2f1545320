"""The workloads that libmadam_amd is timed on, from one small call to the largest solves.

Every case runs through the public Python entry points on a synthetic ring scan
(60 s spin, 85 deg opening angle, 1 deg/hour precession, 100 Hz): a sky of white
noise per pixel plus white and 1/f detector noise.  A case is a dict of plain
values; the keys are

  kind      oneshot   run(): host arrays in, host maps out, one handle per call
            solve     FP64 Madam.solve on a handle that keeps its pointing, then
                      maps() and baselines()
            newscan   set_pointing, solve and maps() of a scan not seen before
            steps     a fixed number of FP64 PCG iterations and the baselines
            batch     Madam.solve_batch and the results of every right-hand side
            serve     a handful of jobs through the request loop
            pointing  the pointing expansion into device buffers
  ndet, nsamp, nside, ncross, nnz, base (s), nperiod, prior, distinct (every
  detector on its own boresight), flags, f32 (FP32 TOD), nrhs, precision, steps, jobs
"""
import math

import numpy as np
import torch

import libmadam_amd

FS = 100.0
SCAN = dict(fsample=FS, spin_period=60.0, prec_period=360 * 3600.0, opening_turns=85.0 / 360.0, lon0_turns=0.0)
SIGMA, FKNEE, ALPHA = 2e-4, 0.05, -1.5
DEFAULTS = dict(ncross=0, nnz=3, base=0.25, nperiod=1, prior=True, distinct=False, flags=False, f32=False, nrhs=1,
                precision=0, steps=0, jobs=0)


def listed():
    return [
        # the smallest call a user makes: a test-sized temperature map, all set-up included
        dict(name="reference_small", kind="oneshot", ndet=4, nsamp=1000, nside=8, ncross=4, nnz=1, base=1.0,
             nperiod=4),
        # a plain polarised destripe from host arrays (4 x 2^20 at Nside 64), no noise prior
        dict(name="plain_host", kind="oneshot", ndet=4, nsamp=2 ** 20, nside=64, base=1.0, prior=False),
        # one realisation of a Monte Carlo loop on a scan of ordinary size
        dict(name="mc_medium", kind="solve", ndet=4, nsamp=2 ** 22, nside=256),
        # the FP64 destripe with noise prior at full size (16 x 2^24 at Nside 512)
        dict(name="mc_large", kind="solve", ndet=16, nsamp=2 ** 24, nside=512, nperiod=2),
        # a flagged scan seen for the first time: pointing set-up, filters, preconditioner, solve
        dict(name="new_scan", kind="newscan", ndet=8, nsamp=2 ** 23, nside=512, base=0.5, nperiod=2, distinct=True,
             flags=True),
        # temperature only, ragged length, the solve on coarser pixels than the map
        dict(name="temperature", kind="solve", ndet=6, nsamp=3000017, nside=256, ncross=128, nnz=1, base=1.0,
             prior=False, distinct=True, flags=True),
        # the mixed-precision solve at Nside 1024 (FP32 TOD, FP64 refinement)
        dict(name="mixed_large", kind="batch", ndet=32, nsamp=2 ** 24, nside=1024, nperiod=4, f32=True, precision=1),
        # sixteen noise realisations of one scan, mixed precision
        dict(name="mixed_batch", kind="batch", ndet=8, nsamp=2 ** 22, nside=256, f32=True, nrhs=16, precision=1),
        # a few realisations in FP64 (the batch is padded to eight)
        dict(name="fp64_batch", kind="batch", ndet=4, nsamp=2 ** 20, nside=128, nrhs=5),
        # PCG iterations alone, ragged, flagged, no shared boresights, map larger than the caches
        dict(name="steps_ragged", kind="steps", ndet=12, nsamp=5000011, nside=1024, nperiod=3, distinct=True,
             flags=True, steps=20),
        # jobs of mixed sizes that arrive together at the request loop
        dict(name="serve", kind="serve", ndet=4, nsamp=2 ** 20, nside=256, f32=True, precision=1, jobs=6),
        # pointing expansion to pixels and weights (16 x 2^22 samples)
        dict(name="pointing", kind="pointing", ndet=16, nsamp=2 ** 22, nside=1024),
    ]


def draw(rng):
    """One more case: sizes spread over the logarithm of the ranges the listed cases span."""
    kind = rng.choice(["oneshot", "solve", "solve", "newscan", "steps", "batch", "batch", "serve", "pointing"])
    size = lambda lo, hi: int(round(2 ** rng.uniform(lo, hi))) | rng.randrange(2)  # noqa: E731
    c = dict(kind=kind, ndet=rng.choice([4, 5, 6, 8, 12, 16]), base=round(rng.uniform(0.25, 1.0), 2),
             nperiod=rng.choice([1, 2, 3]), prior=rng.random() < 0.7, distinct=rng.random() < 0.4,
             flags=rng.random() < 0.4)
    if kind == "oneshot":
        c.update(ndet=rng.choice([4, 8]), nsamp=size(15, 20), nside=rng.choice([16, 32, 64]), flags=False,
                 distinct=False)
    elif kind == "pointing":
        c = dict(kind=kind, ndet=rng.choice([1, 3, 8, 16, 32]), nsamp=size(14, 22), nside=rng.choice([64, 256, 1024]))
    elif kind == "serve":
        c = dict(kind=kind, ndet=4, nsamp=size(18, 20), nside=rng.choice([64, 128, 256]), f32=True, precision=1,
                 jobs=rng.choice([4, 5, 6]))
    elif kind == "batch":
        c.update(ndet=rng.choice([4, 6, 8]), nsamp=size(18, 22), nside=rng.choice([64, 128, 256]),
                 nrhs=rng.choice([1, 2, 5, 8, 16]), precision=rng.choice([0, 1, 1]), f32=rng.random() < 0.6)
    else:
        c.update(nsamp=size(18, 23), nside=rng.choice([64, 128, 256, 512, 1024]))
        if rng.random() < 0.25:
            c.update(nnz=1)
        if rng.random() < 0.25:
            c.update(ncross=c["nside"] // 2)
        if kind == "steps":
            c.update(steps=rng.choice([10, 20]))
    return c


# ------------------------------------------------------------------ inputs


def _full(case):
    return {**DEFAULTS, **case}


def _detectors(c):
    """Four polarisation angles; horns of four detectors, or one boresight each."""
    angles = (0.0, 0.125, 0.25, 0.375)
    if c["distinct"]:
        return [dict(psi_turns=angles[j % 4], open_offset_turns=j * 0.05 / 360.0, spin_offset_turns=j * 0.0011)
                for j in range(c["ndet"])]
    return [dict(psi_turns=angles[j % 4], open_offset_turns=(j // 4) * 0.1 / 360.0, spin_offset_turns=0.0)
            for j in range(c["ndet"])]


def _first_sample(seed):
    return (seed % 1009) * 5011


def _pointing(c, seed):
    """pix int32 [ndet][nsamp] and weights float32 [ndet][nsamp][nnz] on the GPU."""
    nd, ns = c["ndet"], c["nsamp"]
    pix = torch.empty(nd, ns, dtype=torch.int32, device="cuda")
    w = torch.empty(nd, ns, 3, dtype=torch.float32, device="cuda")
    torch.cuda.synchronize()
    libmadam_amd.expand_pointing_device(SCAN, _detectors(c), c["nside"], _first_sample(seed), ns, pix, w)
    if c["nnz"] == 1:
        w = torch.ones(nd, ns, dtype=torch.float32, device="cuda")
    if c["flags"]:
        # about 1 % of the samples in bursts of half a second, and single ones
        g = torch.Generator(device="cuda").manual_seed(seed + 77)
        for d in range(nd):
            burst = torch.rand(ns // 50 + 1, generator=g, device="cuda") < 0.01
            bad = burst.repeat_interleave(50)[:ns] | (torch.rand(ns, generator=g, device="cuda") < 0.002)
            pix[d][bad] = -1
    return pix, w


def _tod(c, pix, w, seed, dtype):
    """Sky (100/5/5 uK white per pixel) plus white and 1/f noise of one realisation."""
    nd, ns, nnz = c["ndet"], c["nsamp"], c["nnz"]
    g = torch.Generator(device="cuda").manual_seed(seed)
    sky = torch.randn(12 * c["nside"] ** 2, 3, generator=g, device="cuda", dtype=torch.float64)
    sky *= torch.tensor([100e-6, 5e-6, 5e-6], device="cuda", dtype=torch.float64)
    nfft = 1 << (ns - 1).bit_length()
    f = torch.fft.rfftfreq(nfft, 1.0 / FS, device="cuda", dtype=torch.float64)
    shape = torch.zeros_like(f)
    shape[1:] = torch.sqrt(1.0 + (f[1:] / FKNEE) ** ALPHA)
    tod = torch.empty(nd, ns, device="cuda", dtype=dtype)
    for d in range(nd):
        white = torch.randn(nfft, generator=g, device="cuda", dtype=torch.float64) * SIGMA
        sig = torch.fft.irfft(torch.fft.rfft(white) * shape, n=nfft)[:ns]
        p = pix[d].clamp(min=0).long()
        if nnz == 1:
            sig = sig + sky[p, 0]
        else:
            for j in range(3):
                sig = sig + sky[p, j] * w[d, :, j]
        tod[d] = sig.to(dtype)
    return tod


def _tables(c):
    freqs = np.logspace(-5, np.log10(FS / 2), 200)
    psd = SIGMA ** 2 / FS * (1.0 + (freqs / FKNEE) ** ALPHA)
    return freqs, psd


def _setup_args(c):
    """The parameters and noise model of one scan, in the order configure() takes them."""
    freqs, psd = _tables(c)
    nd, ns = c["ndet"], c["nsamp"]
    pars = dict(base_first=c["base"], fsample=FS, nside_map=c["nside"], nside_cross=c["ncross"] or c["nside"],
                nside_submap=min(16, c["ncross"] or c["nside"]), kfilter=bool(c["prior"]), info=0)
    periods = (np.arange(c["nperiod"]) * (ns // c["nperiod"])).astype(np.int64)
    dets = ["det%02d" % j for j in range(nd)]
    return (pars, dets, np.full(nd, 1.0 / SIGMA ** 2), np.arange(ns) / FS, periods, np.ones(nd, np.int64),
            np.zeros(nd), freqs, np.tile(psd, nd))


def _handle(c):
    m = libmadam_amd.Madam(0)
    m.configure(*_setup_args(c), c["nnz"])
    return m


def _job_cases(c):
    return [dict(c, nsamp=max(c["nsamp"] >> (j % 3), 4096), nside=max(c["nside"] >> (j % 2), 8), prior=j % 2 == 0,
                 base=0.25 + 0.15 * j) for j in range(c["jobs"])]


def prepare(case, seed):
    c = _full(case)
    torch.cuda.init()
    kind = c["kind"]
    if kind == "pointing":
        pix = torch.empty(c["ndet"], c["nsamp"], dtype=torch.int32, device="cuda")
        w = torch.empty(c["ndet"], c["nsamp"], 3, dtype=torch.float32, device="cuda")
        torch.cuda.synchronize()
        return dict(kind=kind, c=c, dets=_detectors(c), first=_first_sample(seed), pix=pix, w=w)
    if kind == "serve":
        jobs = []
        for j, jc in enumerate(_job_cases(c)):
            pix, w = _pointing(jc, seed + j)
            tod = _tod(jc, pix, w, seed + j, torch.float32)
            jobs.append((_setup_args(jc), pix, w, tod))
        torch.cuda.synchronize()
        return dict(kind=kind, c=c, jobs=jobs, server=libmadam_amd.Server(0, 200e9, 4))
    pix, w = _pointing(c, seed)
    if kind == "batch":
        tod = torch.empty(c["nrhs"], c["ndet"], c["nsamp"], device="cuda",
                          dtype=torch.float32 if c["f32"] else torch.float64)
        for r in range(c["nrhs"]):
            tod[r] = _tod(c, pix, w, seed + 1000003 * r, tod.dtype)
    else:
        tod = _tod(c, pix, w, seed, torch.float64)
    torch.cuda.synchronize()
    if kind == "oneshot":
        return dict(kind=kind, c=c, args=_setup_args(c), pix=pix.cpu().numpy().reshape(-1),
                    w=w.cpu().numpy().reshape(-1), tod=tod.cpu().numpy().reshape(-1))
    m = _handle(c)
    if kind != "newscan":
        m.set_pointing(pix, w, on_device=True)
    if kind == "steps":
        m.solve(tod, on_device=True)
    return dict(kind=kind, c=c, m=m, pix=pix, w=w, tod=tod)


# ------------------------------------------------------------------ one pass


def run(state):
    kind, c = state["kind"], state["c"]
    if kind == "pointing":
        libmadam_amd.expand_pointing_device(SCAN, state["dets"], c["nside"], state["first"], c["nsamp"], state["pix"],
                                            state["w"])
        return dict(pix=state["pix"], w=state["w"])
    if kind == "serve":
        srv = state["server"]
        ids = []
        for (pars, dets, wd, ts, per, npsd, pst, pfr, pv), pix, w, tod in state["jobs"]:
            ids.append(srv.submit(pars, wd, ts, pix, w, tod, per, npsd, pst, pfr, pv, nnz=c["nnz"],
                                  precision=c["precision"], on_device=True))
        out = []
        for j in ids:
            srv.wait(j)
            r = srv.result(j)
            srv.release(j)
            out.append({k: r[k] for k in ("map", "binmap", "hits", "aa")})
        return out
    if kind == "oneshot":
        pars, dets, wd, ts, per, npsd, pst, pfr, pv = state["args"]
        r = libmadam_amd.run(pars, dets, wd, ts, state["pix"], state["w"], state["tod"], per, npsd, pst, pfr, pv)
        return {k: r[k] for k in ("map", "binmap", "hits", "cc", "mask", "aa")}
    m = state["m"]
    if kind == "batch":
        m.solve_batch(state["tod"], precision=c["precision"], on_device=True)
        out = []
        for r in range(c["nrhs"]):
            b = m.batch_result(r)
            out.append({k: b[k] for k in ("map", "binmap", "aa", "yba")})
        return out
    if kind == "steps":
        m.iterate(c["steps"], restart=True)
        return m.baselines()
    if kind == "newscan":
        m.set_pointing(state["pix"], state["w"], on_device=True)
        m.solve(state["tod"], on_device=True)
        return m.maps()
    m.solve(state["tod"], on_device=True)
    out = m.maps()
    out.update(m.baselines())
    return out


# ------------------------------------------------------------------ what a pass cannot do without


def work(case):
    """Bytes: the pointing (an index, and two weights where there is polarisation) and the TOD once, the maps
    and baselines out once; for the fixed PCG steps the pointing on both sides of each step and the vectors of
    the recurrence.  A solve iterates until its residual meets the limit, so its floor here is the one pass
    that every destriping takes at least."""
    c = _full(case)
    if c["kind"] == "serve":
        jobs = [work(dict(j, kind="newscan")) for j in _job_cases(c)]
        return {k: sum(j[k] for j in jobs) for k in ("bytes", "flops")}
    n = c["ndet"] * c["nsamp"]
    nmap = c["nnz"]
    if c["kind"] == "pointing":
        return {"bytes": 16.0 * n, "flops": 150.0 * n}
    npix = 12 * c["nside"] ** 2
    nb = n / max(1.0, round(c["base"] * FS))
    rec = 12 if nmap == 3 else 4
    if c["kind"] == "steps":
        return {"bytes": float(c["steps"] * (2 * rec * n + 12 * 8 * nb + 8 * 4 * npix)),
                "flops": float(c["steps"] * n * (4 * nmap + 4))}
    tod = 4 if c["f32"] else 8
    hit = min(npix, n)
    out = c["nrhs"] * (16 * nmap * npix + 16 * nb) + (0 if c["kind"] == "batch" else npix * (16 + 8 * nmap * nmap))
    start = (4 + 4 * nmap) if c["kind"] in ("oneshot", "newscan") else rec
    return {"bytes": float(start * n + c["nrhs"] * tod * n + out),
            "flops": float(c["nrhs"] * n * (8 * nmap + 4) + 60 * hit)}


def tolerance(case):
    """FP64: the same PCG with its sums in another order differs by up to 2e-13 (pixels near the condition
    limit by 1e-10).  Mixed precision: two FP32 inner solves that both meet the limit on the FP64 residual
    differ by up to 2e-5 with a noise prior and by 1e-3 without one, where the operator is worse conditioned."""
    c = _full(case)
    if c["kind"] == "pointing":
        return "exact"
    if c["precision"] == 1:
        return {"rel": 1e-4, "max": 1e-3} if c["prior"] and c["kind"] != "serve" else {"rel": 4e-3, "max": 0.1}
    return {"rel": 1e-11, "max": 1e-8}


# ------------------------------------------------------------------ the same in plain torch, 64 bits

MOST_SAMPLES = 20_000_000   # of all right-hand sides together: beyond it exact() would take too long


class _Problem:
    """The normal equations of one scan: (F^T W Z F + C_a^-1) a = F^T W Z d."""

    def __init__(self, c, pix, w):
        self.c = c
        nd, ns, nmap = c["ndet"], c["nsamp"], c["nnz"]
        self.nmap = nmap
        self.npix = 12 * c["nside"] ** 2
        self.ncross = 12 * (c["ncross"] or c["nside"]) ** 2
        self.ndeg = self.npix // self.ncross
        self.dw = 1.0 / SIGMA ** 2
        dn = round(c["base"] * FS)
        length = [ns // c["nperiod"]] * (c["nperiod"] - 1)
        length.append(ns - sum(length))
        self.noba = [(n - 1) // dn + 1 for n in length]
        base = torch.cat([torch.arange(n, device="cuda") // dn + sum(self.noba[:i]) for i, n in enumerate(length)])
        self.nbase = sum(self.noba)
        self.nb = nd * self.nbase
        b = (base[None, :] + torch.arange(nd, device="cuda")[:, None] * self.nbase).reshape(-1)
        self.ok = pix.reshape(-1) >= 0
        self.pix = pix.reshape(-1)[self.ok].long()
        self.b = b[self.ok]
        self.w = w.reshape(-1, nmap)[self.ok].double()
        self.q = self.pix // self.ndeg
        cc = self._matrices(self.pix, self.npix)
        self.map_inv = self._invert(cc, np.float32(1e-6).item())
        cross = cc.reshape(self.ncross, self.ndeg, nmap, nmap).sum(1) if self.ndeg > 1 else cc
        self.cross_inv = self._invert(cross, np.float32(1e-3).item())
        self.good = (self.cross_inv != 0).any(-1).any(-1)
        # samples in rejected pixels take no part in F
        use = self.good[self.q]
        self.fq, self.fb, self.fw = self.q[use], self.b[use], self.w[use]
        self.use = use
        self.nna = self._sum(self.fb, torch.full_like(self.fb, 1, dtype=torch.float64), self.nb) * self.dw
        self.fcov = self._filter() if c["prior"] else None

    @staticmethod
    def _sum(index, v, n):
        return torch.zeros(n, dtype=torch.float64, device="cuda").index_add_(0, index, v)

    def _matrices(self, pix, npix):
        cc = torch.zeros(npix, self.nmap, self.nmap, dtype=torch.float64, device="cuda")
        for i in range(self.nmap):
            for j in range(i, self.nmap):
                cc[:, i, j] = cc[:, j, i] = self._sum(pix, self.w[:, i] * self.w[:, j], npix) * self.dw
        return cc

    @staticmethod
    def _invert(cc, limit):
        if cc.shape[-1] == 1:
            return torch.where(cc > 0, 1.0 / cc, torch.zeros_like(cc))
        a, b, d = cc[:, 0, 0], cc[:, 0, 1], cc[:, 0, 2]
        e, f, h = cc[:, 1, 1], cc[:, 1, 2], cc[:, 2, 2]
        adj = torch.stack([e * h - f * f, d * f - b * h, b * f - d * e, d * f - b * h, a * h - d * d, b * d - a * f,
                           b * f - d * e, b * d - a * f, a * e - b * b], -1).reshape(-1, 3, 3)
        det = a * adj[:, 0, 0] + b * adj[:, 0, 1] + d * adj[:, 0, 2]
        # eigenvalues of a symmetric 3 x 3 matrix from its characteristic polynomial
        m = (a + e + h) / 3
        p = (((a - m) ** 2 + (e - m) ** 2 + (h - m) ** 2 + 2 * (b * b + d * d + f * f)) / 6).sqrt()
        r = ((a - m) * ((e - m) * (h - m) - f * f) - b * (b * (h - m) - f * d) + d * (b * f - (e - m) * d))
        phi = torch.arccos((r / (2 * p ** 3).clamp(min=1e-300)).clamp(-1, 1)) / 3
        big = m + 2 * p * torch.cos(phi)
        small = m + 2 * p * torch.cos(phi + 2 * math.pi / 3)
        keep = (big > 0) & (small / big.clamp(min=1e-300) >= limit)
        inv = adj / torch.where(keep, det, torch.ones_like(det))[:, None, None]
        return torch.where(keep[:, None, None], inv, torch.zeros_like(inv))

    def _filter(self):
        """Power spectrum of the baseline offsets, aliased and weighted by the baseline window, inverted."""
        nof = 1
        while nof < max(2 * max(self.noba), 4):
            nof *= 2
        if nof < 101:                  # wide enough for the widest preconditioner
            nof = 128
        freqs, psd = _tables(self.c)
        lf, lp = np.log(freqs), np.log(psd)
        margin = float(np.float32(1e-6))

        def interp(f):
            lx = np.log(np.where(f > 0, f, 1.0))
            j = np.clip(np.searchsorted(lf, lx) - 1, 0, len(lf) - 2)
            t = (lx - lf[j]) / (lf[j + 1] - lf[j])
            return np.where(f > 0, np.exp(lp[j] * (1 - t) + lp[j + 1] * t), 0.0)

        plateau = interp(np.array([FS / 2]))[0]

        def spec(f):
            v = interp(f)
            return np.where(v > plateau * (1 + margin), v - plateau, v * margin)

        fa = FS / round(self.c["base"] * FS)
        i = np.arange(nof // 2 + 1)
        asp = np.zeros(nof // 2 + 1)
        for k in range(3):
            for at in (k * fa + i * fa / nof, k * fa + (nof - i) * fa / nof):
                asp += spec(at) * np.sinc(at / fa) ** 2
        fcov = 1.0 / (fa * asp)
        fcov[0] = 0.0
        self.nof = nof
        return torch.from_numpy(fcov).cuda()

    def _segments(self, x, spectrum, project):
        """Convolution with a spectrum on every (detector, period), less the segment mean on both sides."""
        x = x.reshape(self.c["ndet"], self.nbase)
        out = torch.empty_like(x)
        at = 0
        for n in self.noba:
            v = x[:, at:at + n]
            mean = v.mean(1, keepdim=True)
            y = torch.fft.irfft(torch.fft.rfft(v - mean, n=self.nof) * spectrum, n=self.nof)[:, :n]
            y = y - y.mean(1, keepdim=True)
            out[:, at:at + n] = y if project else y + mean / self.nna.mean()
            at += n
        return out.reshape(-1)

    def _binned(self, inv, q, w, v, n):
        m = torch.stack([self._sum(q, w[:, j] * v, n) for j in range(self.nmap)], -1) * self.dw
        return (inv @ m[..., None])[..., 0]

    def operator(self, p):
        v = p[self.fb]
        m = self._binned(self.cross_inv, self.fq, self.fw, v, self.ncross)
        v = v - (self.fw * m[self.fq]).sum(-1)
        y = self._sum(self.fb, v, self.nb) * self.dw
        return y + self._segments(p, self.fcov, True) if self.fcov is not None else y

    def precondition(self, r):
        if self.fcov is None:
            return torch.where(self.nna > 0, r / self.nna.clamp(min=1e-300), torch.zeros_like(r))
        return self._segments(r, 1.0 / (self.fcov + self.nna.mean()), False)

    def null_weights(self):
        """M 1 of the solver's preconditioner M.  A constant added to all baselines is not determined by the
        data; a PCG that starts from zero leaves a with (M 1) . a = 0."""
        if self.fcov is None:
            return self.nna
        inv = torch.fft.irfft(self.fcov, n=self.nof).cpu().numpy()
        total = float((inv[:self.nof // 2] ** 2).sum())
        out = self.nna.clone().reshape(self.c["ndet"], self.nbase)
        at = 0
        for n in self.noba:
            width = 10
            while width < min(n, 100) and not (inv[:min(width, n)] ** 2).sum() > np.float32(1 - 1e-5) * total:
                width += 10
            width = min(width, n, 100)
            if width <= 50 and (inv[:width] ** 2).sum() > np.float32(1 - 1e-5) * total:
                c = np.concatenate([[0.0], np.cumsum(inv[1:width])])
                k = np.arange(n)
                row = inv[0] + c[np.minimum(k, width - 1)] + c[np.minimum(n - 1 - k, width - 1)]
                out[:, at:at + n] += torch.from_numpy(row).cuda()
            at += n
        return out.reshape(-1)

    def solve(self, tod):
        d = tod.reshape(-1)[self.ok].double()
        rhs_q = self._binned(self.cross_inv, self.q, self.w, d, self.ncross)
        fd = d[self.use] - (self.fw * rhs_q[self.fq]).sum(-1)
        yba = self._sum(self.fb, fd, self.nb) * self.dw
        a = torch.zeros_like(yba)
        r = yba.clone()
        z = self.precondition(r)
        p, rz, rr0 = z.clone(), r @ z, r @ r
        for _ in range(400):
            ap = self.operator(p)
            alpha = rz / (p @ ap)
            a += alpha * p
            r -= alpha * ap
            if (r @ r) / rr0 < 1e-24:
                break
            z = self.precondition(r)
            new = r @ z
            p = z + (new / rz) * p
            rz = new
        u = self.null_weights()
        a -= (u @ a) / u.sum()
        if self.fcov is None:
            a = torch.where(self.nna > 0, a, torch.zeros_like(a))
        binmap = self._binned(self.map_inv, self.pix, self.w, d, self.npix)
        dmap = self._binned(self.map_inv, self.pix, self.w, d - a[self.b], self.npix)
        shape = (self.c["ndet"], self.nbase)
        return dict(map=dmap, binmap=binmap, aa=a.reshape(shape), yba=yba.reshape(shape))


def exact(case, seed):
    c = _full(case)
    kind = c["kind"]
    if kind in ("serve", "steps") or c["ndet"] * c["nsamp"] * c["nrhs"] > MOST_SAMPLES:
        return None
    torch.cuda.init()
    if kind == "pointing":
        return dict(pix=None, w=_exact_weights(c, seed))
    pix, w = _pointing(c, seed)
    prob = _Problem(c, pix, w)
    nmap = c["nnz"]
    if kind == "batch":
        out = []
        for r in range(c["nrhs"]):
            tod = _tod(c, pix, w, seed + 1000003 * r, torch.float32 if c["f32"] else torch.float64)
            s = prob.solve(tod)
            out.append({k: s[k] for k in ("map", "binmap", "aa", "yba")})
        return out
    s = prob.solve(_tod(c, pix, w, seed, torch.float64))
    cc = prob.map_inv.reshape(prob.npix, nmap, nmap)
    if kind == "oneshot":
        return dict(map=s["map"], binmap=s["binmap"], hits=None, cc=cc, mask=None, aa=s["aa"])
    if kind == "newscan":
        return dict(map=s["map"], binmap=s["binmap"], hits=None, cc=cc, mask=None, crit=None)
    return dict(map=s["map"], binmap=s["binmap"], hits=None, cc=cc, mask=None, crit=None, aa=s["aa"], yba=s["yba"],
                nna=prob.nna.reshape(c["ndet"], -1))


def _exact_weights(c, seed):
    """(1, cos 2 psi, sin 2 psi) of the ring scan, from the attitude's rotations in 64 bits."""
    t = (torch.arange(c["nsamp"], device="cuda", dtype=torch.float64) + _first_sample(seed)) / FS
    w = torch.empty(c["ndet"], c["nsamp"], 3, dtype=torch.float64, device="cuda")
    lon = 2 * math.pi * (t / SCAN["prec_period"])
    zero = torch.zeros_like(t)
    for j, d in enumerate(_detectors(c)):
        spin = 2 * math.pi * (t / SCAN["spin_period"] + d["spin_offset_turns"])
        opening = 2 * math.pi * (SCAN["opening_turns"] + d["open_offset_turns"])
        psi = 2 * math.pi * d["psi_turns"]
        axis = torch.stack([torch.cos(lon), torch.sin(lon), zero])
        side = torch.stack([-torch.sin(lon), torch.cos(lon), zero])
        north = torch.stack([zero, zero, zero + 1])
        bore = math.cos(opening) * axis + math.sin(opening) * (torch.sin(spin) * side + torch.cos(spin) * north)
        along = torch.cos(spin) * side - torch.sin(spin) * north
        pol = math.cos(psi) * along + math.sin(psi) * torch.linalg.cross(bore, along, dim=0)
        rho = (bore[0] ** 2 + bore[1] ** 2).sqrt()
        south = torch.stack([bore[2] * bore[0] / rho, bore[2] * bore[1] / rho, -rho])
        east = torch.stack([-bore[1] / rho, bore[0] / rho, zero])
        u, v = (pol * south).sum(0), (pol * east).sum(0)
        w[j, :, 0] = 1.0
        w[j, :, 1] = (u * u - v * v) / (u * u + v * v)
        w[j, :, 2] = -2 * u * v / (u * u + v * v)
    return w
