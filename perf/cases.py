"""The work a user of the search has the device do, as cases that can be timed.

A case is a dict of plain values; "kind" says which path it takes:

  block   one data block through one ddplan row, call by call, as the drop-in
          runs it (push, dedispersion, boxcar, thresholded points or maps).
          The beam is in steady state: the same block is pushed every pass, so
          the input is periodic and every pass has the same outputs.
  search  a short observation through several rows, one graph launch per
          block, every point in pinned host memory.
  cuts    zdot and kadaneF on a batch of candidate cutouts, in place.
  front   a raw 8-bit block through the front end's statistics, its
          equalisation, zdot and kadaneF, as the search's RFI chain runs them.
  grid    the refinement grid (dedispersion tree and matched filter).
  grad    the differentiable S/N, forward and backward through autograd.
  steps   the two calls that gradient refinement is made of: the coarse grid
          and the adjoint of runs of evaluations with second derivatives.
"""
from __future__ import annotations

import math

import numpy as np
import torch

KDM = 4.148741601e3
THRE = 7.0

# bands and sampling of the configurations: fbot, ftop (MHz), tsamp (s)
BANDS = {
    "test": (1200.0, 1500.0, 1e-3),
    "lband": (1200.0, 1500.0, 98.304e-6),
    "wide": (856.0, 1712.0, 76.56e-6),
    "fast": (1000.0, 1500.0, 16e-6),
}


def _block(name, band, nchans, nsub, ndump, dms, ddm, ndm, overlap, minw, maxw, dtype, out):
    c = dict(kind="block", band=band, nchans=nchans, nsub=nsub, ndump=ndump, dms=dms, ddm=ddm, ndm=ndm,
             overlap=overlap, minw=minw, maxw=maxw, dtype=dtype, out=out)
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # the smallest call: a test-sized beam, where launches and latency count
        _block("block 64ch u8", "test", 64, 8, 512, 0.0, 2.0, 40, 0.25, 1e-3, 0.05, "u8", "points"),
        # an ordinary single-row search of a 1024-channel 8-bit beam, 2 s blocks
        _block("block 1024ch u8", "lband", 1024, 32, 20345, 0.0, 1.0, 1000, 0.1, 1e-4, 0.1, "u8", "points"),
        # the production beam's first row on raw 8-bit blocks equalised on the device
        _block("block 4096ch raw", "wide", 4096, 64, 26123, 0.0, 0.5, 1000, 0.1, 1e-4, 0.1, "raw", "points"),
        # the drop-in on front-end floats with the S/N and width maps kept for its readers
        _block("block 4096ch f32 maps", "wide", 4096, 64, 26123, 500.0, 2.0, 500, 0.1, 1e-4, 0.1, "f32", "maps"),
        # a 2048-channel beam's high-DM row in the reference's own summation order
        _block("block 2048ch exact", "wide", 2048, 64, 26123, 1500.0, 5.0, 300, 0.1, 1e-4, 0.1, "u8", "exact"),
        # high time resolution: the longest row of the 16 us plan, the largest block
        _block("block 4096ch 16us u8", "fast", 4096, 64, 31250, 0.0, 0.2, 2500, 0.0, 16e-6, 5e-3, "u8", "points"),
        # the production beam, three rows, 12 blocks of 2 s as graph launches
        dict(name="search 4096ch", kind="search", band="wide", nchans=4096, ndump=26123, nblocks=12,
             rows="0,0.5,1000,64;500,2,500,64;1500,5,300,128", overlap=0.1, minw=1e-4, maxw=0.1),
        # replot's cleaning of the candidates of an observation
        dict(name="cuts 1024x512", kind="cuts", ncut=1024, nchan=1024, nbin=512, td=4, fd=2, thr=5.0),
        # the RFI chain on one production block
        dict(name="front 4096ch", kind="front", nchan=4096, nsamp=26123, td=1, fd=1, ktd=4, kfd=2, thr=7.0),
        # replot's refinement grid
        dict(name="grid 1024x512", kind="grid", ncut=512, nchan=1024, nbin=512, maps=False),
        # S/N and its gradients for a batch of candidates
        dict(name="grad 1024x512", kind="grad", ncut=512, nchan=1024, nbin=512, need_x=False),
        # the calls of gradient refinement on the same cutouts
        dict(name="steps 1024x512", kind="steps", ncut=128, nchan=1024, nbin=512, run=48, ndm=9, nt0=9),
    ]


def _logint(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["block", "block", "block", "block", "search", "cuts", "front", "grid", "grad", "steps"])
    if kind in ("block", "search"):
        band = rng.choice(["lband", "wide", "wide", "fast"])
        cps = rng.choice([8, 16, 20, 32, 50, 64])
        nsub = _logint(rng, 8, 128)
        while cps * nsub > 4096:
            nsub = nsub // 2
        nchans = cps * nsub
        ndump = _logint(rng, 1500, 31250)
        overlap = rng.choice([0.0, 0.1, 0.25])
        tsamp = BANDS[band][2]
        maxw = min(0.1 if band != "fast" else 5e-3, 0.2 * ndump * tsamp)
        # DM steps as the configurations pair them with their bands
        dms, ddm = rng.choice({"lband": [(0.0, 1.0), (100.0, 2.0)], "fast": [(0.0, 0.2), (500.0, 1.0)],
                               "wide": [(0.0, 0.5), (500.0, 2.0), (1500.0, 5.0)]}[band])
        ndm = _logint(rng, 24, 1000)
        minw = 16e-6 if band == "fast" else 1e-4
        if kind == "block":
            return _block("", band, nchans, nsub, ndump, dms, ddm, ndm, overlap, minw, maxw,
                          rng.choice(["u8", "u8", "f32", "raw"]), rng.choice(["points", "points", "maps", "exact"]))
        ndm2 = _logint(rng, 24, 500)
        rows = "%g,%g,%d,%d;%g,%g,%d,%d" % (dms, ddm, ndm, nsub, dms + ddm * ndm, 2 * ddm, ndm2, nsub)
        return dict(kind="search", band=band, nchans=nchans, ndump=ndump, nblocks=rng.randint(6, 12), rows=rows,
                    overlap=overlap, minw=minw, maxw=maxw)
    if kind == "front":
        td, fd = rng.choice([(1, 1), (1, 1), (2, 1), (1, 2), (4, 2)])
        return dict(kind="front", nchan=_logint(rng, 256, 4096), nsamp=_logint(rng, 1000, 26123), td=td, fd=fd,
                    ktd=rng.choice([1, 2, 4, 8]), kfd=rng.choice([1, 2, 4]), thr=7.0)
    nchan, nbin = _logint(rng, 64, 1024), _logint(rng, 64, 1024)
    if kind == "cuts":
        return dict(kind="cuts", ncut=_logint(rng, 4, 1024), nchan=nchan, nbin=nbin, td=rng.choice([1, 2, 4, 8]),
                    fd=rng.choice([1, 2, 4]), thr=5.0)
    if kind == "grid":
        return dict(kind="grid", ncut=_logint(rng, 4, 256), nchan=nchan, nbin=nbin, maps=rng.random() < 0.5)
    if kind == "grad":
        return dict(kind="grad", ncut=_logint(rng, 4, 512), nchan=nchan, nbin=nbin, need_x=rng.random() < 0.3)
    nbin = max(64, nbin // 4 * 4)
    return dict(kind="steps", ncut=_logint(rng, 4, 128), nchan=nchan, nbin=nbin, run=rng.choice([6, 20, 48]),
                ndm=rng.choice([5, 9]), nt0=rng.choice([5, 9, 17]))


# ------------------------------------------------------------------ inputs
def _freqs(nchans, fbot, ftop):
    return ftop - (np.arange(nchans) + 0.5) * ((ftop - fbot) / nchans)


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _noise_block(g, rng, n, freqs, tsamp, pulses, repeat=True):
    """[n][C] u8: N(128, 12^2), 0.5% of the channels at five times that, dispersed pulses (dm, sample, sigma, amplitude)."""
    C = freqs.size
    sd = torch.full((C,), 12.0, device="cuda")
    sd[torch.from_numpy(rng.choice(C, max(1, C // 200), replace=False)).cuda()] = 60.0
    x = torch.randn((n, C), generator=g, device="cuda") * sd + 128.0
    t = torch.arange(n, device="cuda", dtype=torch.float32)[:, None]
    for dm, t0, sig, amp in pulses:
        d = torch.from_numpy(KDM * dm * (1 / freqs ** 2 - 1 / freqs.max() ** 2) / tsamp).cuda().float()
        u = t - (t0 + d)
        if repeat:
            u = torch.remainder(u + n / 2, n) - n / 2
        x += amp * torch.exp(-0.5 * (u / sig) ** 2)
    return x.round_().clamp_(0, 255).to(torch.uint8)


def _pulse(rng, case, C, dms, ddm, ndm):
    """A pulse of S/N about 14 (less what the DM step smears) somewhere in the row, a narrow one or a few widths of the ladder long."""
    tsamp = BANDS[case["band"]][2]
    dm = dms + ddm * ndm * float(rng.uniform(0.2, 0.9))
    lo = math.log(max(case["minw"], tsamp))
    sig = max(1.0, math.exp(float(rng.uniform(lo, max(lo, math.log(case["maxw"] / 4))))) / tsamp / 4)
    amp = 14.0 * 12.0 / math.sqrt(C * 2.5 * sig)
    return dm, float(rng.uniform(0, case["ndump"])), sig, amp


def _block_input(case, seed):
    """The block a pass pushes (and the front end's offset and gain of it for raw blocks)."""
    rng = np.random.default_rng(seed)
    fbot, ftop, tsamp = BANDS[case["band"]]
    freqs = _freqs(case["nchans"], fbot, ftop)
    x = _noise_block(_gen(seed), rng, case["ndump"], freqs, tsamp,
                     [_pulse(rng, case, case["nchans"], case["dms"], case["ddm"], case["ndm"])])
    if case["dtype"] == "u8":
        return freqs, x, None
    xf = x.double()
    off = xf.mean(0).float()
    gain = (1.0 / (xf - xf.mean(0)).square().mean(0).sqrt()).float()
    if case["dtype"] == "f32":
        return freqs, (x.float() - off) * gain, None
    return freqs, x, (off, gain)


def _points(v, keys, cap):
    """A block's points in arrays of the caller's own size, the number found first."""
    out = {k: np.zeros(cap, v[k].dtype) for k in keys}
    n = min(cap, v.size)
    for k in keys:
        out[k][:n] = v[k][:n]
    out["n"] = v.size
    return out


class _View:
    """A device buffer of the library as a torch tensor, without a copy."""

    def __init__(self, ptr, shape, typestr):
        self.__cuda_array_interface__ = dict(shape=shape, typestr=typestr, data=(ptr, False), version=2, strides=None)


def _view(ptr, shape, typestr):
    return torch.as_tensor(_View(ptr, shape, typestr), device="cuda")


def _rows(case):
    out = []
    for r in case["rows"].split(";"):
        dms, ddm, ndm, nsub = r.split(",")
        out.append((float(dms), float(ddm), int(ndm), int(nsub)))
    return out


def _cutouts(case, seed):
    """Unit-variance cutouts, 3% of channels zero, one dispersed pulse each
    around the centre, dedispersed at a DM that is a little off."""
    n, nchan, nbin = case["ncut"], case["nchan"], case["nbin"]
    rng, g = np.random.default_rng(seed), _gen(seed)
    f = np.linspace(1500.0, 1200.0 + 300.0 / nchan, nchan)
    tbin = 98.304e-6
    dl = torch.from_numpy(KDM * (1 / f ** 2 - 1 / f.max() ** 2) / tbin).cuda()
    dm = rng.uniform(50, 1500, n)
    ctr = torch.from_numpy(nbin / 2 + rng.uniform(-8, 8, n)).cuda()
    sig = torch.from_numpy(np.exp(rng.uniform(math.log(2.0), math.log(max(3.0, nbin / 8)), n))).cuda()
    amp = torch.from_numpy(rng.uniform(8, 40, n)).cuda() / torch.sqrt(2.5 * sig * nchan)
    x = torch.randn((n, nchan, nbin), generator=g, device="cuda")
    t = torch.arange(nbin, device="cuda", dtype=torch.float32)
    dmt = torch.from_numpy(dm).cuda()
    for c0 in range(0, n, 64):
        s = slice(c0, min(n, c0 + 64))
        at = (ctr[s, None] + dmt[s, None] * dl).float()
        u = torch.remainder(t - at[:, :, None] + nbin / 2, float(nbin)) - nbin / 2
        x[s] += amp[s, None, None].float() * torch.exp(-0.5 * (u / sig[s, None, None].float()) ** 2)
    mask = torch.rand((n, nchan), generator=g, device="cuda") < 0.03
    x[mask] = 0.0
    return f, tbin, x, (~mask).float().contiguous(), dm, ctr, sig, rng


def _dirty(case, seed):
    """Cutouts with zero-DM interference of per-channel gain and a narrowband burst each."""
    n, nchan, nbin = case["ncut"], case["nchan"], case["nbin"]
    g = _gen(seed)
    x = torch.randn((n, nchan, nbin), generator=g, device="cuda")
    x += torch.rand((n, nchan, 1), generator=g, device="cuda") * 6 * torch.randn((n, 1, nbin), generator=g, device="cuda")
    j = torch.randint(0, nchan, (n,), generator=g, device="cuda")
    x[torch.arange(n, device="cuda"), j, nbin // 4:nbin // 2] += 6.0
    return x


def _raw(case, seed):
    """A raw 8-bit block with interference common to the channels and bursts in a few of them."""
    ni, ci = case["nsamp"] * case["td"], case["nchan"] * case["fd"]
    rng, g = np.random.default_rng(seed), _gen(seed)
    x = torch.randn((ni, ci), generator=g, device="cuda") * 12 + 128
    x += torch.randn((ni, 1), generator=g, device="cuda") * 3 * torch.rand((1, ci), generator=g, device="cuda")
    for _ in range(8):
        j, t = int(rng.integers(ci)), int(rng.integers(max(1, ni - ni // 16)))
        x[t:t + ni // 16, j] += 24
    return x.round_().clamp_(0, 255).to(torch.uint8)


def _grad_input(case, seed):
    f, tbin, x, w, dm, ctr, sig, rng = _cutouts(case, seed)
    n = case["ncut"]
    fl = lambda v: torch.as_tensor(v, dtype=torch.float32, device="cuda").contiguous()  # noqa: E731
    return (f, tbin, x, w, fl(dm + rng.uniform(-0.3, 0.3, n)), fl(ctr + torch.from_numpy(rng.uniform(-2, 2, n)).cuda()),
            fl(2.5 * sig), fl(rng.uniform(0.5, 1.5, n)))


def _steps_input(case, seed):
    f, tbin, x, w, dm, ctr, sig, rng = _cutouts(case, seed)
    n, run = case["ncut"], case["run"]
    fl = lambda v: torch.as_tensor(v, dtype=torch.float32, device="cuda").contiguous()  # noqa: E731
    dme = fl((dm[:, None] + rng.uniform(-0.5, 0.5, (n, run))).reshape(-1))
    t0 = fl((ctr.cpu().numpy()[:, None] + rng.uniform(-4, 4, (n, run))).reshape(-1))
    wd = fl((2.5 * sig.cpu().numpy()[:, None] * rng.uniform(0.7, 1.4, (n, run))).reshape(-1))
    widths = fl(np.geomspace(1.0, case["nbin"] / 2, 16))
    return f, tbin, x, w, dme, t0, wd, fl(dm - 0.25 * (case["ndm"] - 1)), fl(ctr - (case["nt0"] - 1)), widths


# --------------------------------------------------------------- the cases
def prepare(case, seed):
    from transientx_amd import Beam, Plan, width_ladder
    from transientx_amd.diff import DiffSNR
    from transientx_amd.refine import Refiner

    kind = case["kind"]
    if kind == "block":
        freqs, x, eq = _block_input(case, seed)
        tsamp = BANDS[case["band"]][2]
        beam = Beam(case["nchans"], case["ndump"], dtype="u8" if case["dtype"] == "u8" else "f32", zero_point=128)
        if eq is not None:
            beam.set_frontend(case["nchans"], 1, 1, eq[0].cpu().numpy(), eq[1].cpu().numpy())
        vwn = width_ladder(tsamp, case["minw"], case["maxw"], 0.1)
        plan = Plan(beam, freqs=freqs, tsamp=tsamp, dms=case["dms"], ddm=case["ddm"], ndm=case["ndm"], vwn=vwn,
                    overlap=case["overlap"], nsub=case["nsub"], store_maps=case["out"] != "points",
                    exact_order=case["out"] == "exact")
        o = plan.info
        t, s, w = plan.device_buffers()
        shp = (o.ndm, o.nsamples)
        st = dict(kind=kind, case=case, beam=beam, plan=plan, block=x, tim=_view(t, shp, "<f4"))
        if case["out"] != "points":
            st.update(mxS=_view(s, shp, "<f4"), mxwn=_view(w, shp, "<i4"))
        torch.cuda.synchronize()
        for _ in range(-(-(o.offset + o.nsamples) // o.ndump)):  # up to the boxcar's gate and a whole window
            beam.push(x)
            plan.dedisp_run()
        beam.sync()
        return st
    if kind == "search":
        rng, g = np.random.default_rng(seed), _gen(seed)
        fbot, ftop, tsamp = BANDS[case["band"]]
        freqs = _freqs(case["nchans"], fbot, ftop)
        rows = _rows(case)
        beam = Beam(case["nchans"], case["ndump"], dtype="u8", zero_point=128)
        vwn = width_ladder(tsamp, case["minw"], case["maxw"], 0.1)
        plans = [Plan(beam, freqs=freqs, tsamp=tsamp, dms=a, ddm=b, ndm=n, vwn=vwn, overlap=case["overlap"],
                      nsub=k, store_maps=False) for a, b, n, k in rows]
        blocks = [_noise_block(g, rng, case["ndump"], freqs, tsamp,
                               [_pulse(rng, case, case["nchans"], *rows[k % len(rows)][:3])] if k % 3 == 0 else [])
                  for k in range(case["nblocks"])]
        cap = 1 << 20
        host = [torch.empty(cap * 24, dtype=torch.uint8, pin_memory=True) for _ in plans]
        torch.cuda.synchronize()
        beam.reset()
        for p, h in zip(plans, host):
            p.session_begin(cap, host=h)
        beam.build_graph(THRE)
        beam.sync()
        return dict(kind=kind, case=case, beam=beam, plans=plans, blocks=blocks, host=host, cap=cap, open=True)
    if kind == "cuts":
        return dict(kind=kind, case=case, x=_dirty(case, seed), wnl=np.zeros(case["ncut"], np.int32))
    if kind == "front":
        return dict(kind=kind, case=case, x=_raw(case, seed))
    if kind == "grid":
        f, tbin, x, w, dm, ctr, sig, rng = _cutouts(case, seed)
        R = Refiner(f, case["nbin"], tbin, 0.1, dedisperse=True, isdedispersed=True, max_batch=256)
        return dict(kind=kind, case=case, R=R, x=x, dm=dm + rng.uniform(-2, 2, case["ncut"]))
    if kind == "grad":
        f, tbin, x, w, dm, t0, wd, gs = _grad_input(case, seed)
        x.requires_grad_(bool(case["need_x"]))
        for v in (w, dm, t0, wd):
            v.requires_grad_(True)
        return dict(kind=kind, case=case, D=DiffSNR(f, case["nbin"], tbin, softness=1.0), x=x, w=w, dm=dm, t0=t0, wd=wd,
                    gs=gs)
    f, tbin, x, w, dme, t0, wd, d0, tz, widths = _steps_input(case, seed)
    return dict(kind=kind, case=case, D=DiffSNR(f, case["nbin"], tbin, softness=1.0), x=x, w=w, dm=dme, t0=t0, wd=wd,
                d0=d0, tz=tz, widths=widths, one=torch.ones_like(dme))


def run(s):
    from transientx_amd import frontend, rfi
    from transientx_amd.diff import refine_snr

    kind, case = s["kind"], s["case"]
    if kind == "block":
        s["beam"].push(s["block"])
        s["plan"].dedisp_run()
        s["plan"].boxcar_run(THRE)
        out = {"tim": s["tim"], **_points(s["plan"].points(), ("idm", "isamp", "S", "wn"), 1 << 14)}
        if case["out"] != "points":
            out.update(mxS=s["mxS"], mxwn=s["mxwn"])
        return out
    if kind == "search":
        beam, plans = s["beam"], s["plans"]
        beam.reset()
        if not s["open"]:
            for p, h in zip(plans, s["host"]):
                p.session_begin(s["cap"], host=h)
        s["open"] = False
        for b in s["blocks"]:
            beam.graph_push(b)
        out = []
        for p in plans:
            v = p.session_end()
            o = np.argsort((v["block"].astype(np.int64) << 48) | (v["idm"].astype(np.int64) << 32) | v["isamp"])
            out.append(_points(v[o], ("block", "idm", "isamp", "S", "wn"), 1 << 16))
        return out
    if kind == "cuts":
        return rfi.kadane_f(rfi.zdot(s["x"]), case["td"], case["fd"], case["thr"], s["wnl"])
    if kind == "front":
        off, gain = frontend.stats(s["x"], case["td"], case["fd"])
        y = frontend.apply(s["x"], case["td"], case["fd"], off, gain)
        rfi.zdot(y, layout="time")
        rfi.kadane_f(y, case["ktd"], case["kfd"], case["thr"], 0, layout="time")
        return {"off": off, "gain": gain, "y": y}
    if kind == "grid":
        r = s["R"].run(s["x"], s["dm"], maps=case["maps"])
        res, maps = r if case["maps"] else (r, ())
        return [{k: np.ascontiguousarray(res[k]) for k in ("maxdmid", "maxtid", "snr", "wn", "width", "dm_maxsnr")},
                *maps]
    if kind == "grad":
        ins = [s["w"], s["dm"], s["t0"], s["wd"]] + ([s["x"]] if case["need_x"] else [])
        S = refine_snr(s["D"], s["x"], s["w"], s["dm"], s["t0"], s["wd"])
        return [S.detach(), *torch.autograd.grad(S, ins, s["gs"])]
    D = s["D"]
    best, idx = D.grid(s["x"], s["w"], s["d0"], s["tz"], case["ndm"], 0.5, case["nt0"], 2.0, s["widths"])
    return [best, idx, *D.adjoint_runs(s["x"], s["w"], s["dm"], s["t0"], s["wd"], s["one"], run=case["run"], second=True)]


def _group(freqs, nsub, ndm):
    cps = freqs.size // nsub
    lo = int(np.argmin(freqs)) // cps
    fr = freqs[lo * cps:(lo + 1) * cps].max()
    dsub = 1 / freqs.min() ** 2 - 1 / fr ** 2
    dband = 1 / freqs.min() ** 2 - 1 / freqs.max() ** 2
    return max(1, min(ndm, 1 + int(math.floor(dband / dsub)) if dsub > 0 else ndm))


def _ladder(case):
    from transientx_amd import width_ladder

    return width_ladder(BANDS[case["band"]][2], case["minw"], case["maxw"], 0.1)


def _row_work(case, ndm, nsub, nblocks):
    fbot, ftop, _ = BANDS[case["band"]]
    C, nd = case["nchans"], case["ndump"]
    N = nd + int(case["overlap"] * nd)
    ndmc = -(-ndm // _group(_freqs(C, fbot, ftop), nsub, ndm))
    return N, float(nblocks) * (C * ndmc * nd + nsub * ndm * N + 2 * len(_ladder(case)) * ndm * N)


def work(case):
    kind = case["kind"]
    if kind == "block":
        N, flops = _row_work(case, case["ndm"], case["nsub"], 1)
        C, nd = case["nchans"], case["ndump"]
        maps = 8 if case["out"] != "points" else 0
        return {"bytes": C * nd * (4 if case["dtype"] == "f32" else 1) + (4 + maps) * case["ndm"] * N, "flops": flops}
    if kind == "search":
        flops = by = 0.0
        for _, _, ndm, nsub in _rows(case):
            N, f = _row_work(case, ndm, nsub, case["nblocks"])
            flops += f
            by += 4.0 * ndm * N * case["nblocks"]  # a row's series, which its boxcar takes
        return {"bytes": by + case["nchans"] * case["ndump"] * case["nblocks"], "flops": flops}
    if kind == "front":
        n = case["nchan"] * case["nsamp"]
        return {"bytes": n * (case["td"] * case["fd"] + 4), "flops": 20.0 * n}
    n = case["ncut"] * case["nchan"] * case["nbin"]
    if kind == "cuts":
        return {"bytes": 8 * n, "flops": 18.0 * n}
    if kind == "grid":
        nrow = 1 << max(1, math.ceil(math.log2(case["nchan"])))
        m = case["ncut"] * nrow * case["nbin"]
        nbox, v = 0, 1
        while v <= case["nbin"] // 2:
            nbox, v = nbox + 1, max(v + 1, int(v * 1.2345679))
        return {"bytes": 4 * n + (12 * m if case["maps"] else 0), "flops": m * (math.log2(nrow) + 8 + 2.0 * nbox)}
    if kind == "grad":
        return {"bytes": 4 * n * (2 if case["need_x"] else 1), "flops": 12.0 * n}
    ev = case["run"] + case["ndm"]
    return {"bytes": 4 * n, "flops": n * (5.0 * ev + 5.0 * case["run"])}


# ------------------------------------------------------- the same in 64 bits
def _lround(v):
    return (np.sign(v) * np.floor(np.abs(v) + 0.5)).astype(np.int64)


def _exact_series(case, freqs, x):
    """tim [ndm][N] of the periodic input x [ndump][C] (float64)."""
    tsamp = BANDS[case["band"]][2]
    C, nsub, ndm, nd = case["nchans"], case["nsub"], case["ndm"], case["ndump"]
    N = nd + int(case["overlap"] * nd)
    cps, g = C // nsub, _group(freqs, nsub, ndm)
    ndmc = -(-ndm // g)
    fref = freqs.reshape(nsub, cps).max(1)
    delay = lambda dm, f: _lround(KDM * dm * (1 / f ** 2 - 1 / freqs.max() ** 2) / tsamp)  # noqa: E731
    gk = np.minimum(g, ndm - g * np.arange(ndmc))
    dmc = case["dms"] + case["ddm"] * (g * np.arange(ndmc) + (gk - 1) / 2.0)
    d1 = delay(dmc[:, None], freqs[None, :]) - np.repeat(delay(dmc[:, None], fref[None, :]), cps, 1)
    d2 = delay((case["dms"] + case["ddm"] * np.arange(ndm))[:, None], fref[None, :])
    w0 = -int(d1.max()) - int(d2.max()) - N
    d1, d2 = torch.from_numpy(d1).cuda(), torch.from_numpy(d2).cuda()
    t = torch.arange(nd, device="cuda")
    xt = x.t().contiguous()
    kc = torch.arange(ndm, device="cuda") // g
    tim = torch.zeros((ndm, N), dtype=torch.float64, device="cuda")
    tw = torch.arange(N, device="cuda")
    for s in range(nsub):
        sub = torch.zeros((ndmc, nd), dtype=torch.float64, device="cuda")
        for j in range(s * cps, (s + 1) * cps):
            sub += xt[j][(t + d1[:, j:j + 1]) % nd]
        flat = sub.reshape(-1)
        for i0 in range(0, ndm, 512):
            i1 = min(ndm, i0 + 512)
            tim[i0:i1] += flat[(kc[i0:i1] * nd)[:, None] + (tw + w0 + d2[i0:i1, s:s + 1]) % nd]
    return tim


def _exact_maps(tim, vwn):
    """The largest S/N over the widths, each in the output range that the reference's vector loop gives it."""
    ndm, N = tim.shape
    out = torch.zeros_like(tim)
    m = tim.mean(1, keepdim=True)
    var = (tim - m).square().mean(1, keepdim=True)
    for i0 in range(0, ndm, 128):
        s = slice(i0, min(ndm, i0 + 128))
        cs = torch.cumsum(tim[s] - m[s], 1)
        for wn in vwn.tolist():
            wl, wh = wn // 2 + 1, (wn - 1) // 2
            n = max(0, N - wh - wl) // 8 * 8
            if n:
                S = (cs[:, wl + wh:wl + wh + n] - cs[:, :n]) / torch.sqrt(wn * var[s])
                out[s, wl:wl + n] = torch.maximum(out[s, wl:wl + n], S)
    return out


def _exact_zdot(x):
    """x [frames][channels][samples], float64."""
    sd = (x - x.mean(2, keepdim=True)).square().mean(2, keepdim=True).sqrt()
    x = (x - x.mean(2, keepdim=True)) / torch.where(sd == 0, torch.ones_like(sd), sd)
    s = x.mean(1, keepdim=True)
    sc = s - s.mean(2, keepdim=True)
    ss = sc.square().sum(2, keepdim=True)
    a = torch.where(ss > 0, (x * sc).sum(2, keepdim=True) / ss, torch.zeros_like(ss))
    return x - x.mean(2, keepdim=True) - a * sc


def _exact_kadane(x, td, fd, thr):
    f, c, n = x.shape
    cd, nd = c // fd, n // td
    d = x[:, :cd * fd, :nd * td].reshape(f, cd, fd, nd, td).sum((2, 4)).reshape(f * cd, nd).t().contiguous()
    y = x[:, :cd * fd].reshape(f * cd, fd, n)
    at = torch.arange(n, device=x.device)
    for sg in (1.0, -1.0):
        best = torch.full((f * cd,), -math.inf, dtype=torch.float64, device=x.device)
        cur, st = torch.zeros_like(best), torch.zeros(f * cd, dtype=torch.int64, device=x.device)
        b0, b1 = st.clone(), st.clone()
        for i in range(nd):
            cur = cur + sg * d[i]
            up = cur > best
            best, b0, b1 = torch.where(up, cur, best), torch.where(up, st, b0), torch.where(up, i, b1)
            low = cur < 0
            cur, st = torch.where(low, 0.0, cur), torch.where(low, i + 1, st)
        hit = best * best / ((b1 - b0 + 1) * (td * fd)) > thr * thr
        zap = hit[:, None] & (at >= (b0 * td)[:, None]) & (at < ((b1 + 1) * td)[:, None])
        y = torch.where(zap[:, None, :], 0.0, y)
    out = x.clone()
    out[:, :cd * fd] = y.reshape(f, cd * fd, n)
    return out


def _profiles(f, tbin, x, w, dm, idx):
    """p(t), dp/dDM and the parts of the weights' gradient for evaluations dm of the cutouts idx."""
    nbin = x.shape[2]
    kf = torch.from_numpy(KDM * (1 / f ** 2 - 1 / f.max() ** 2) / tbin).cuda()
    t = torch.arange(nbin, device="cuda")
    tau = dm.double()[:, None] * kf
    d = torch.floor(tau)
    a = (tau - d)[:, :, None]
    i0 = (t + d.long()[:, :, None]) % nbin
    xe = x[idx].double()
    x0, x1 = torch.gather(xe, 2, i0), torch.gather(xe, 2, (i0 + 1) % nbin)
    xs = (1 - a) * x0 + a * x1
    q = torch.einsum("ejt,ej->et", x1 - x0, w[idx].double() * kf)
    return xs, torch.einsum("ejt,ej->et", xs, w[idx].double()), q, i0, a


def _template(t0, wd, nbin):
    t = torch.arange(nbin, device="cuda", dtype=torch.float64)
    dl = torch.remainder(t - t0[..., None] + nbin / 2, float(nbin)) - nbin / 2
    g = torch.sigmoid(dl + wd[..., None] / 2) - torch.sigmoid(dl - wd[..., None] / 2)
    return g - g.mean(-1, keepdim=True)


def _exact_grid(case, f, tbin, x, dm):
    """S/N of the strongest point of each cutout (and the maps) of the dedispersion tree and matched filter."""
    n, nchan, nbin = x.shape
    nrow = 1 << max(1, math.ceil(math.log2(nchan)))
    lv = nrow.bit_length() - 1
    fP = np.concatenate([f, f[0] + (f[1] - f[0]) * np.arange(nchan, nrow)])
    rng_ = nbin * tbin / (KDM * (1 / f.min() ** 2 - 1 / f.max() ** 2))
    dms = np.maximum(0.0, dm - rng_ / 2)
    ddm = (dm + rng_ / 2 - dms) / nrow
    rev = np.array([int(format(k, "0%db" % lv)[::-1], 2) for k in range(nrow)])
    sh = _lround(KDM * dm[:, None] * (1 / f ** 2 - 1 / f.max() ** 2) / tbin) % nbin
    t = torch.arange(nbin, device="cuda")
    A = torch.zeros((n, nrow, nbin), dtype=torch.float64, device="cuda")
    A[:, :nchan] = torch.gather(x.double(), 2, (t + torch.from_numpy(sh).cuda()[:, :, None]) % nbin)
    for l in range(lv):
        k = np.arange(nrow)
        half = 1 << l
        j0 = (k >> (l + 1)) << (l + 1)
        a, b = j0 + (k & (half - 1)), j0 + half + (k & (half - 1))
        dtrial = dms[:, None] + rev[k & (2 * half - 1)][None, :] * ddm[:, None] - dm[:, None]
        s = _lround(KDM * dtrial * (1 / fP[j0 + half] ** 2 - 1 / fP[j0] ** 2) / tbin) % nbin
        A = A[:, a] + torch.gather(A[:, b], 2, (t + torch.from_numpy(s).cuda()[:, :, None]) % nbin)
    A = A[:, torch.from_numpy(rev).cuda()].contiguous()
    v = [1]
    while (u := max(v[-1] + 1, int(np.float32(v[-1]) * np.float32(1 / (1 - float(np.float32(0.1))) ** 2)))) <= nbin // 2:
        v.append(u)
    m = A.mean(2, keepdim=True)
    var = (A - m).square().mean(2, keepdim=True)
    cs = torch.cumsum(torch.cat([A, A], 2) - m, 2)
    S = torch.zeros_like(A)
    for wn in v:
        wl, wh = wn // 2 + 1, (wn - 1) // 2
        i = torch.where(t >= wl, t, t + nbin)
        S = torch.maximum(S, torch.where(var > 0, (cs[:, :, i + wh] - cs[:, :, i - wl]) / torch.sqrt(wn * var), 0.0))
    return S.reshape(n, -1).max(1).values, A, S


def exact(case, seed):
    kind = case["kind"]
    if kind == "block":
        freqs, x, eq = _block_input(case, seed)
        x = (x.double() - eq[0].double()) * eq[1].double() if eq is not None else \
            x.double() - 128.0 if case["dtype"] == "u8" else x.double()
        tim = _exact_series(case, freqs, x)
        out = {"tim": tim, **dict.fromkeys(("idm", "isamp", "S", "wn", "n"))}
        if case["out"] != "points":
            out.update(mxS=_exact_maps(tim, _ladder(case)), mxwn=None)
        return out
    if kind == "search":
        return None  # lists of points above a threshold: which they are is not a number
    if kind == "cuts":
        x = _dirty(case, seed)
        out = torch.empty(x.shape, dtype=torch.float64, device="cuda")
        for c0 in range(0, case["ncut"], 256):
            y = _exact_zdot(x[c0:c0 + 256].double())
            out[c0:c0 + 256] = _exact_kadane(y, case["td"], case["fd"], case["thr"])
        return out
    if kind == "front":
        x, n, c = _raw(case, seed), case["nsamp"], case["nchan"]
        y = x.reshape(n, case["td"], c, case["fd"]).sum((1, 3)).double()
        off = y.mean(0)
        gain = 1 / (y - off).square().mean(0).sqrt()
        y = _exact_zdot(((y - off) * gain).t()[None].contiguous())
        y = _exact_kadane(y, case["ktd"], case["kfd"], case["thr"])
        return {"off": off, "gain": gain, "y": y[0].t().contiguous()}
    if kind == "grid":
        f, tbin, x, w, dm, ctr, sig, rng = _cutouts(case, seed)
        dm = dm + rng.uniform(-2, 2, case["ncut"])
        top, maps = [], [[], []]
        for c0 in range(0, case["ncut"], 32):
            s, A, S = _exact_grid(case, f, tbin, x[c0:c0 + 32], dm[c0:c0 + 32])
            top.append(s)
            if case["maps"]:
                maps[0].append(A)
                maps[1].append(S)
        res = dict.fromkeys(("maxdmid", "maxtid", "wn", "width", "dm_maxsnr"))
        res["snr"] = torch.cat(top)
        return [res, torch.cat(maps[0]), torch.cat(maps[1]), None] if case["maps"] else [res]
    if kind == "grad":
        f, tbin, x, w, dm, t0, wd, gs = _grad_input(case, seed)
        outs = [[] for _ in range(6 if case["need_x"] else 5)]
        for c0 in range(0, case["ncut"], 32):
            e = torch.arange(c0, min(case["ncut"], c0 + 32), device="cuda")
            xs, p, q, i0, a = _profiles(f, tbin, x, w, dm[e], e)
            tt, ww = t0[e].double().requires_grad_(True), wd[e].double().requires_grad_(True)
            g = _template(tt, ww, case["nbin"])
            G = g / (g.norm(dim=1) * w[e].double().norm(dim=1))[:, None]
            S, u = (G * p).sum(1), gs[e].double()
            gt, gw = torch.autograd.grad((S * u).sum(), [tt, ww])
            G, S = G.detach(), S.detach()
            wj = w[e].double()
            got = [S, u[:, None] * (torch.einsum("et,ejt->ej", G, xs) - S[:, None] * wj / wj.square().sum(1, keepdim=True)),
                   u * (G * q).sum(1), gt, gw]
            if case["need_x"]:
                Ge = (u[:, None, None] * wj[:, :, None]) * G[:, None, :]
                got.append(torch.zeros_like(xs).scatter_add_(2, i0, (1 - a) * Ge).scatter_add_(2, (i0 + 1) % case["nbin"], a * Ge))
            for k, v in zip(outs, got):
                k.append(v)
        return [torch.cat(v) for v in outs]
    f, tbin, x, w, dme, t0, wd, d0, tz, widths = _steps_input(case, seed)
    n, nbin, run_ = case["ncut"], case["nbin"], case["run"]
    best, outs = [], [[] for _ in range(6)]
    trial = torch.arange(case["ndm"], device="cuda") * 0.5
    ts = torch.arange(case["nt0"], device="cuda") * 2.0
    for c in range(n):
        wn = w[c].double().norm()
        one = torch.zeros(case["ndm"], dtype=torch.long, device="cuda") + c
        _, p, _, _, _ = _profiles(f, tbin, x, w, d0[c].double() + trial, one)
        g = _template((tz[c].double() + ts)[:, None], widths.double()[None, :], nbin).reshape(-1, nbin)
        best.append(((p @ (g / g.norm(dim=1, keepdim=True)).t()) / wn).max(1).values)
        e = slice(c * run_, (c + 1) * run_)
        one = torch.zeros(run_, dtype=torch.long, device="cuda") + c
        _, p, q, _, _ = _profiles(f, tbin, x, w, dme[e], one)
        tt, ww = t0[e].double().requires_grad_(True), wd[e].double().requires_grad_(True)
        g = _template(tt, ww, nbin)
        G = g / (g.norm(dim=1, keepdim=True) * wn)
        S, Q = (G * p).sum(1), (G * q).sum(1)
        gt, gw = torch.autograd.grad(S.sum(), [tt, ww], create_graph=True)
        gtt = torch.autograd.grad(gt.sum(), tt, retain_graph=True)[0]
        gdt = torch.autograd.grad(Q.sum(), tt)[0]
        for k, v in zip(outs, (S, Q, gt, gw, gtt, gdt)):
            k.append(v.detach())
    return [torch.stack(best), None, *[torch.cat(v) for v in outs]]
