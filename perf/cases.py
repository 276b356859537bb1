"""Performance cases of the GPP sigma library: what its users have it evaluate,
through the public Python binding, from the smallest call to the largest.

The sizes are this repository's own: the mini-app's published jobs (512 2 N 20
with ncouls 800, 1600 and 3200), the CPU configuration 512/2/4096/409, the
benchmark shape 512/2/32768/1638, the large single instance
1536/8/65536/3276 with 16 frequencies, the batch of 64 uneven instances, and
the smoke call.  Inputs have the benchmark distributions (aqs re/im ~U(-1,1),
I_eps ~U(-0.5,0.5), wtilde re ~U(0.5,5) im ~U(-0.05,0.05), vcoul ~U(0.1,10),
sorted distinct random inv_igp_index), drawn on the GPU from the seed.

A case names the entry point in "call":
  sigma      Context.bind_device once, Context.sigma per pass
  launchers  the three reference-compatible device launchers, outputs zeroed
             and accumulated on the null stream
  batch      Batch over caller-owned device inputs, Batch.sigma per pass
"""
import math
import os
import sys

import numpy as np
import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(_ROOT, "doe-csfg-hackathon_amd"))

import pygpp  # noqa: E402

_DEV = "cuda"


def _case(call, form, nb, nv, nc, ng, nf, center=4.0, dw=1.0, acht=False, groups=0, slab=0, count=0, span=0):
    """groups: rows of band-dependent frequencies (0: one shared row).  slab:
    ranks the G' columns are divided over, one of them evaluated (0: all).
    count, span: a batch's instances and the seed of their sizes (the sizes
    given are then the largest ones)."""
    return {"call": call, "form": form, "nb": nb, "nv": nv, "nc": nc, "ng": ng, "nf": nf, "center": center, "dw": dw,
            "acht": acht, "groups": groups, "slab": slab, "count": count, "span": span}


def listed():
    cases = {
        # the smallest call: the smoke evaluation, every output wanted
        "smoke_all": _case("sigma", "factored-f64", 24, 2, 1000, 50, 3, acht=True),
        # the mini-app's small job in the factored form: latency and launches
        "job_small": _case("sigma", "factored-f64", 512, 2, 800, 40, 3),
        # the mini-app's medium job in the direct form, the drop-in for its
        # timed loop (every output)
        "job_med_direct": _case("sigma", "direct", 512, 2, 1600, 80, 3, acht=True),
        # the mini-app's big job as the CUDA driver runs it: device arrays and
        # the three launchers
        "job_big_launchers": _case("launchers", "direct", 512, 2, 3200, 160, 3),
        # a validation run: the reference's operation order, odd sizes, two
        # passes of frequencies
        "strict_odd": _case("sigma", "direct-strict", 131, 5, 2477, 123, 7, dw=0.5, acht=True),
        # the CPU configuration, every output from the factored form
        "cpu_shape_all": _case("sigma", "factored-f64", 512, 2, 4096, 409, 3, acht=True),
        # energies that depend on the band: 8 groups of bands, the higher ones
        # at negative frequencies
        "band_rows": _case("sigma", "factored-f64", 512, 8, 8192, 409, 3, groups=8),
        # one rank's columns of the benchmark shape divided over 8 ranks
        "rank_slab": _case("sigma", "factored-f64", 512, 2, 32768, 1638, 3, slab=8),
        # the benchmark shape
        "bench": _case("sigma", "factored-f64", 512, 2, 32768, 1638, 3),
        # the benchmark shape with the integer split of the Gram product
        "bench_i8": _case("sigma", "factored-ozaki-i8", 512, 2, 32768, 1638, 3),
        # the large instance, 16 frequencies
        "large_16f": _case("sigma", "factored-f64", 1536, 8, 65536, 3276, 16, dw=0.25),
        # 64 uneven instances in one pass (3 to 32 frequencies, 2 to 8 occupied bands)
        "batch_64": _case("batch", "factored-f64", 1024, 8, 16384, 819, 32, count=64, span=4),
    }
    return [dict(c, name=k) for k, c in cases.items()]


def draw(rng):
    def logint(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["factored", "factored", "all", "direct", "strict", "launchers", "rows", "slab", "i8", "batch"])
    nv, nf = rng.randint(0, 9), rng.choice([1, 2, 3, 3, 3, 4, 5, 7, 8, 11, 13, 16, 19, 24])
    nb = max(logint(24, 1200), nv + 4)
    dw = 1.0 if nf <= 3 else 4.0 / nf
    if kind in ("direct", "strict", "launchers"):
        # every update is evaluated: at most about 4e9 of them
        nc = logint(400, 8000)
        ng = max(1, nc // rng.choice([8, 10, 20, 20, 37]))
        nf = 3 if kind == "launchers" else nf
        while nb * ng * nc * nf > 4e9:
            nc = int(nc * 0.8)
            ng = max(1, int(ng * 0.8))
        form = {"direct": "direct", "strict": "direct-strict", "launchers": "direct"}[kind]
        return _case("launchers" if kind == "launchers" else "sigma", form, nb, nv, nc, ng, nf, dw=dw, acht=True)
    if kind == "batch":
        return _case("batch", rng.choice(["factored-f64", "factored-f64", "factored-ozaki-i8"]), logint(160, 1024), 8,
                     logint(2500, 16384), 819, 32, count=rng.randint(3, 48), span=rng.randint(5, 1 << 20))
    nc = logint(400, 50000)
    ng = max(1, nc // rng.choice([8, 10, 20, 20, 37]))
    while nb * ng * nc > 1.2e11:  # the Gram product stays below the large instance's
        ng = int(ng * 0.8)
    if kind == "rows":
        return _case("sigma", "factored-f64", nb, nv, min(nc, 12000), min(ng, 600), nf, dw=dw, groups=rng.randint(1, 12))
    if kind == "slab":
        return _case("sigma", "factored-f64", nb, nv, nc, max(ng, 8), nf, dw=dw, slab=rng.choice([2, 4, 8]))
    return _case("sigma", "factored-ozaki-i8" if kind == "i8" else "factored-f64", nb, nv, nc, ng, nf, dw=dw,
                 acht=kind == "all")


def _instances(case):
    """The problems of a case: (nb, nv, nc, ng, nf, center, dw) each."""
    if not case["count"]:
        return [tuple(case[k] for k in ("nb", "nv", "nc", "ng", "nf", "center", "dw"))]
    r = np.random.default_rng(case["span"])
    out = []
    for _ in range(case["count"]):
        nb = int(r.integers(128, case["nb"] + 1))
        nv = int(r.integers(2, case["nv"] + 1))
        nc = int(r.integers(2048, case["nc"] + 1))
        nf = int(r.integers(3, case["nf"] + 1))
        out.append((nb, nv, nc, nc // 20, nf, 4.0, 2.0 / (nf - 1)))  # the frequency window [3, 5]
    return out


def _wx(nf, center, dw):
    return [max(center + dw * (iw - 0.5 * (nf - 1)), 1e-6) for iw in range(nf)]


def _band_rows(case):
    """wx_bands [nb][nf], as the mini-app forms them with an energy per band:
    e_lk - e(band) + dw (iw - 1); occupied bands lie in the first group."""
    nb, nf, g = case["nb"], case["nf"], case["groups"]
    rows = np.zeros((nb, nf))
    for n in range(nb):
        k = 0 if n < case["nv"] else n * g // nb
        rows[n] = [10.0 - (6.0 + 1.37 * k) + case["dw"] * (iw - 0.5 * (nf - 1)) for iw in range(nf)]
    return rows


def _slab(case):
    """Columns [j0, j1) of the evaluated rank: the second one."""
    if not case["slab"]:
        return 0, case["ng"]
    per = -(-case["ng"] // case["slab"])
    return per, min(2 * per, case["ng"])


def _inputs(inst, seed):
    """One problem's arrays on the GPU."""
    nb, nv, nc, ng, nf, center, dw = inst
    g = torch.Generator(device=_DEV)
    g.manual_seed(seed)

    def uniform(shape, lo_re, hi_re, lo_im, hi_im):
        x = torch.rand(*shape, 2, dtype=torch.float64, device=_DEV, generator=g)
        x[..., 0].mul_(hi_re - lo_re).add_(lo_re)
        x[..., 1].mul_(hi_im - lo_im).add_(lo_im)
        return torch.view_as_complex(x)

    t = {
        "aqsmtemp": uniform((nb, nc), -1.0, 1.0, -1.0, 1.0),
        "aqsntemp": uniform((nb, nc), -1.0, 1.0, -1.0, 1.0),
        "I_eps_array": uniform((ng, nc), -0.5, 0.5, -0.5, 0.5),
        "wtilde_array": uniform((ng, nc), 0.5, 5.0, -0.05, 0.05),
        "vcoul": torch.rand(nc, dtype=torch.float64, device=_DEV, generator=g) * 9.9 + 0.1,
        "inv_igp_index": torch.randperm(nc, device=_DEV, generator=g)[:ng].sort().values.to(torch.int32),
        "wx_array": torch.tensor(_wx(nf, center, dw), dtype=torch.float64, device=_DEV),
    }
    return t


def _problem(inst):
    nb, nv, nc, ng, nf, _, _ = inst
    return pygpp.Problem(nb, nv, nc, ng, nf)


def prepare(case, seed):
    insts = _instances(case)
    tens = [_inputs(inst, 1000 * seed + i) for i, inst in enumerate(insts)]
    ptrs = [{k: v.data_ptr() for k, v in t.items()} for t in tens]
    torch.cuda.synchronize()  # the library works on its context's stream
    st = {"case": case, "tens": tens}
    if case["call"] == "launchers":
        st["lib"] = pygpp.load()
        st["out"] = {
            "achtemp_re": torch.zeros(3, dtype=torch.float64, device=_DEV),
            "achtemp_im": torch.zeros(3, dtype=torch.float64, device=_DEV),
            "asxtemp": torch.zeros(3, dtype=torch.complex128, device=_DEV),
            "acht_n1_loc": torch.zeros(case["nb"], dtype=torch.complex128, device=_DEV),
            "achstemp_re": torch.zeros(1, dtype=torch.float64, device=_DEV),
            "achstemp_im": torch.zeros(1, dtype=torch.float64, device=_DEV),
        }
        return st
    st["ctx"] = pygpp.Context(0)
    if case["call"] == "batch":
        st["batch"] = pygpp.Batch(st["ctx"], [_problem(i) for i in insts], device_inputs=ptrs)
        return st
    st["ctx"].bind_device(_problem(insts[0]), ptrs[0])
    if case["groups"]:
        st["ctx"].set_band_frequencies(_band_rows(case))
    if case["slab"]:
        st["ctx"].set_columns(*_slab(case))
    return st


def run(st):
    case = st["case"]
    if case["call"] == "batch":
        outs = st["batch"].sigma(case["form"])
        return {"achtemp": np.concatenate([o["achtemp"] for o in outs]),
                "asxtemp": np.concatenate([o["asxtemp"] for o in outs]),
                "achstemp": np.array([o["achstemp"] for o in outs])}
    if case["call"] == "launchers":
        lib, o = st["lib"], st["out"]
        p = {k: v.data_ptr() for k, v in st["tens"][0].items()}
        for t in o.values():
            t.zero_()
        q = {k: v.data_ptr() for k, v in o.items()}
        nb, nv, nc, ng = (case[k] for k in ("nb", "nv", "nc", "ng"))
        status = lib.d_reduce_achstemp(nb, p["inv_igp_index"], nc, p["aqsmtemp"], p["aqsntemp"], p["I_eps_array"],
                                       q["achstemp_re"], q["achstemp_im"], ng, p["vcoul"])
        status = status or lib.d_till_nvband(nv, ng, nc, p["inv_igp_index"], p["wx_array"], p["wtilde_array"],
                                             p["aqsmtemp"], p["aqsntemp"], p["I_eps_array"], q["asxtemp"],
                                             p["vcoul"], q["acht_n1_loc"], q["achtemp_re"], q["achtemp_im"], 1.0)
        status = status or lib.d_noFlagOCCSolver(nb, nv, ng, nc, p["inv_igp_index"], p["wx_array"],
                                                 p["wtilde_array"], p["aqsmtemp"], p["aqsntemp"], p["I_eps_array"],
                                                 p["vcoul"], q["achtemp_re"], q["achtemp_im"], q["acht_n1_loc"])
        if status:
            raise RuntimeError(lib.gpp_last_error().decode())
        return o
    return st["ctx"].sigma(case["form"], acht_n1_loc=case["acht"])


def work(case):
    """Bytes: every input a pass depends on read once (aqsmtemp only at the
    column indices), every output written once.  Operations: the direct form
    evaluates each update (33 per unoccupied, 62 per occupied one); the
    factored form needs the band sum as a complex product (8 per
    multiplication and addition), the pole factors (27 per element and
    frequency) and, for acht_n1_loc, a second product."""
    nbytes = flops = 0
    for nb, nv, nc, ng, nf, _, _ in _instances(case):
        if case["slab"]:
            j0, j1 = _slab(case)
            ng = j1 - j0
        nbytes += 16 * (nb * nc + nb * ng + 2 * ng * nc) + 8 * nc + 4 * ng + 16 * (2 * nf + nb + 1)
        if case["form"].startswith("direct"):
            flops += ng * nc * nf * (33 * (nb - nv) + 62 * nv)
        else:
            groups = max(1, case["groups"])
            flops += 8 * ng * nc * nb * (2 if case["acht"] else 1) + 27 * groups * ng * nc * nf
    return {"bytes": nbytes, "flops": flops}


def _pole_factors(wx, wt, ie, occupied):
    """delw*I_eps of one frequency and, for occupied bands, (sch, ssx) of the
    mini-app's solver with its branch tests in its order of operations, on
    real and imaginary parts."""
    wr, wi = wt.real, wt.imag
    dr, di = wx - wr, -wi
    den = dr * dr + di * di
    rden = 1.0 / den
    delr, deli = (wr * dr + wi * di) * rden, (wi * dr - wr * di) * rden
    delw = torch.complex(delr, deli)
    p = delw * ie
    if not occupied:
        return p, None, None
    delw2 = delr * delr + deli * deli
    wt2 = wt * wt
    om2 = wt2 * ie
    b1 = (den > 0.25) & (delw2 < 1.0 / (1e-6 * 4.0))
    b2 = ~b1 & (delw2 > 1e-6)
    cden = 4.0 * wt2 * (delw + 0.5)
    ssx = torch.where(b1, om2 / (wx * wx), torch.where(b2, -om2 * delw / cden, torch.zeros_like(om2)))
    if wx < 0:
        ssx = torch.where(ssx.abs() > 4.0 * ie.abs(), torch.zeros_like(ssx), ssx)
    return p, torch.where(b1, p, torch.zeros_like(p)), ssx


def _exact_one(case, inst, t):
    nb, nv, nc, ng, nf, center, dw = inst
    j0, j1 = _slab(case) if case["slab"] else (0, ng)
    idx = t["inv_igp_index"].to(torch.int64)[j0:j1]
    am, an, vc = t["aqsmtemp"], t["aqsntemp"], t["vcoul"]
    vcj = vc[idx]
    bg = am[:, idx].conj().resolve_conj()
    rows = _band_rows(case) if case["groups"] else np.array([_wx(nf, center, dw)] * nb)
    uniq, member = np.unique(rows, axis=0, return_inverse=True)
    member = member.reshape(-1)
    ach = torch.zeros(nf, dtype=torch.complex128, device=_DEV)
    asx = torch.zeros(nf, dtype=torch.complex128, device=_DEV)
    acht = torch.zeros(nb, dtype=torch.complex128, device=_DEV)
    acht_iw = 2 if nf > 2 else nf - 1
    step = max(1, min(j1 - j0, (1 << 25) // nc))
    for g, row in enumerate(uniq):
        bands = np.nonzero(member == g)[0]
        occ = torch.from_numpy(bands[bands < nv]).to(_DEV)
        un = torch.from_numpy(bands[bands >= nv]).to(_DEV)
        for a in range(0, j1 - j0, step):
            b = min(a + step, j1 - j0)
            wt, ie = t["wtilde_array"][j0 + a:j0 + b], t["I_eps_array"][j0 + a:j0 + b]
            mu = bg[un, a:b].t().contiguous() @ an[un]
            mo = bg[occ, a:b].t().contiguous() @ an[occ] if len(occ) else None
            w = vcj[a:b, None]
            for iw in range(nf):
                p, sch, ssx = _pole_factors(float(row[iw]), wt, ie, mo is not None)
                f = p * mu
                if mo is not None:
                    f = f + sch * mo
                    asx[iw] += ((ssx * mo).sum(1, keepdim=True) * w).sum()
                ach[iw] += 0.5 * (f.sum(1, keepdim=True) * w).sum()
                if iw == acht_iw and (case["acht"] or case["form"].startswith("direct")):
                    acht[un] += 0.5 * (bg[un, a:b] * (an[un] @ (w * p).t().contiguous())).sum(1)
                    if len(occ):
                        acht[occ] += 0.5 * (bg[occ, a:b] * (an[occ] @ (w * sch).t().contiguous())).sum(1)
    schs = -t["I_eps_array"][j0:j1].gather(1, idx[:, None])[:, 0]
    schs = torch.where(schs.abs() > 1e-6, schs, torch.zeros_like(schs))
    achs = ((bg * an[:, idx]).sum(0) * schs * vcj * 0.5).sum()
    return ach, asx, acht, achs


def exact(case, seed):
    got = []
    for i, inst in enumerate(_instances(case)):
        t = _inputs(inst, 1000 * seed + i)
        got.append(_exact_one(case, inst, t))
        del t
    ach, asx, acht, achs = got[0]
    if case["call"] == "batch":
        return {"achtemp": torch.cat([x[0] for x in got]), "asxtemp": torch.cat([x[1] for x in got]),
                "achstemp": torch.stack([x[3] for x in got])}
    if case["call"] == "launchers":
        return {"achtemp_re": ach.real.contiguous(), "achtemp_im": ach.imag.contiguous(), "asxtemp": asx,
                "acht_n1_loc": acht, "achstemp_re": achs.real.reshape(1), "achstemp_im": achs.imag.reshape(1)}
    return {"achtemp": ach, "asxtemp": asx, "acht_n1_loc": acht if case["acht"] else None, "achstemp": achs}
