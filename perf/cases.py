"""Performance cases of the spherical harmonic transforms.

Every case goes through the package's public entry points: batched plans on
device memory, convolution batches, and the drop-ins on host arrays.  A pass
of a transform case is one forward call and one inverse call on separate
inputs, so both directions' results come back whole.  A REAL synthesis and a
convolution return the real plane: the imaginary plane of a real field is
rounding noise, which no caller reads.

Case keys
  kind    "plan"         Plan.forward + Plan.inverse, device tensors
          "conv_batch"   ConvBatch.run: convolutions of uneven bandwidth
          "dropin_pair"  InvFSTSemiMemo + FSTSemiMemo on host arrays
          "dropin_conv"  ConvOn2SphereSemiMemo on host arrays
  bw      bandwidth (the grid is 2bw x 2bw); the largest one of a conv batch
  fields  fields per call (requests of a conv batch)
  prec    "fp64", "mixed" or "split" (S2AMD_FP64, _MIXED, _SPLIT_BF16)
  real    REAL data format (else COMPLEX)
  cutoff  first order of the naive branch (bw: all seminaive)
"""
import math

import numpy as np
import torch

import s2kit_amd as S
from s2kit_amd import synth

PREC = {"fp64": S.FP64, "mixed": S.MIXED, "split": S.SPLIT_BF16}


def _plan(name, bw, fields, prec, real=False, cutoff=None):
    return {"name": name, "kind": "plan", "bw": bw, "fields": fields, "prec": prec, "real": real,
            "cutoff": bw if cutoff is None else cutoff}


def listed():
    return [
        # an S2kit program that kept its own loop: one field, host buffers, its own tables
        {"name": "dropin_pair_bw64", "kind": "dropin_pair", "bw": 64, "fields": 1, "prec": "fp64", "real": False,
         "cutoff": 64},
        # S2kit's convolution example (filter matching on the sphere) on host buffers
        {"name": "dropin_conv_bw128", "kind": "dropin_conv", "bw": 128, "fields": 1, "prec": "fp64", "real": True,
         "cutoff": 128},
        # one small field per call: the latency of an iterative solver's inner step
        _plan("fp64_bw64_x1", 64, 1, "fp64"),
        # one large field per call: a time step of a spectral model
        _plan("fp64_bw512_x1", 512, 1, "fp64"),
        # an ensemble of real fields at moderate resolution
        _plan("fp64_real_bw128_x64", 128, 64, "fp64", real=True),
        # a large batch in full precision
        _plan("fp64_bw256_x1024", 256, 1024, "fp64"),
        # the same batch in the form meant for throughput
        _plan("mixed_bw256_x1024", 256, 1024, "mixed"),
        # a real-valued training batch (spherical CNN layers)
        _plan("mixed_real_bw128_x512", 128, 512, "mixed", real=True),
        # high resolution in the split-BF16 form
        _plan("split_bw512_x64", 512, 64, "split"),
        # a grid that is not a power of two (510 = 2*3*5*17 rings), hybrid cutoff as S2kit's own test uses
        _plan("fp64_bw255_x256_cut64", 255, 256, "fp64", cutoff=64),
        # a ring length with a large prime factor (526 = 2*263)
        _plan("fp64_bw263_x32", 263, 32, "fp64"),
        # requests of many bandwidths at once: a serving batch
        {"name": "conv_batch_x512", "kind": "conv_batch", "bw": 512, "fields": 512, "prec": "mixed", "real": True,
         "cutoff": 512},
    ]


# grid samples of the largest listed case
_MOST = 1024 * 512 * 512


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    u = rng.random()
    if u < 0.08:
        bw = _log_int(rng, 16, 128)
        return {"kind": "dropin_pair", "bw": bw, "fields": 1, "prec": "fp64", "real": rng.random() < 0.5,
                "cutoff": bw if rng.random() < 0.7 else bw // 4}
    if u < 0.14:
        bw = _log_int(rng, 16, 128)
        return {"kind": "dropin_conv", "bw": bw, "fields": 1, "prec": "fp64", "real": True, "cutoff": bw}
    if u < 0.22:
        return {"kind": "conv_batch", "bw": rng.choice([128, 256, 512]), "fields": _log_int(rng, 16, 512),
                "prec": rng.choice(["mixed", "fp64"]), "real": True, "cutoff": 512}
    prec = rng.choice(["fp64", "fp64", "fp64", "mixed", "mixed", "split"])
    if prec == "split":
        bw = rng.choice([32, 64, 128, 256, 512])
    elif rng.random() < 0.5:
        bw = rng.choice([16, 32, 64, 128, 256, 512, 1024] if prec == "fp64" else [32, 64, 128, 256, 512])
    else:
        bw = _log_int(rng, 16 if prec == "fp64" else 32, 512)
    # ring lengths that are not powers of two cost up to three times as much per sample
    share = 1 if bw & (bw - 1) == 0 else 4
    fields = _log_int(rng, 1, max(1, min(2048, _MOST // (4 * bw * bw) // share)))
    cutoff = bw
    if prec == "fp64" and rng.random() < 0.3:
        cutoff = rng.choice([bw // 4, bw // 2, 0])
    return {"kind": "plan", "bw": bw, "fields": fields, "prec": prec, "real": rng.random() < 0.4, "cutoff": cutoff}


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _dev():
    return torch.device("cuda:0" if torch.cuda.is_available() else "cpu")


def _grids(bw, fields, real, seed, dev):
    """Correlated random fields on the 2bw x 2bw grid: a plane spectrum
    falling as 1/(1+|k|)^2, plus white noise a tenth as strong (measurement
    noise, and content past the bandwidth)."""
    n = 2 * bw
    g = torch.Generator(device=dev)
    g.manual_seed(seed)
    k = torch.fft.fftfreq(n, 1.0 / n, dtype=torch.float64, device=dev)
    amp = n / (1.0 + (k[:, None] ** 2 + k[None, :] ** 2).sqrt()) ** 2
    re = torch.empty((fields, n, n), dtype=torch.float64, device=dev)
    im = torch.empty((fields, n, n), dtype=torch.float64, device=dev)
    step = max(1, (1 << 26) // (n * n))
    for f in range(0, fields, step):
        m = min(step, fields - f)
        z = torch.randn((m, n, n, 2), generator=g, dtype=torch.float64, device=dev)
        z = torch.fft.ifft2(torch.view_as_complex(z) * amp, norm="ortho")
        w = 0.1 * torch.randn((2, m, n, n), generator=g, dtype=torch.float64, device=dev)
        re[f:f + m] = z.real + w[0]
        if real:
            im[f:f + m] = 0
        else:
            im[f:f + m] = z.imag + w[1]
    return re, im


def _neg_rows(bw):
    """Coefficient slots of orders 1 .. bw-1 and of their mirror orders, and the signs (-1)^m."""
    l, m = synth.degrees(bw), synth.orders(bw)
    at = {(a, b): i for i, (a, b) in enumerate(zip(l.tolist(), m.tolist()))}
    pos = np.flatnonzero(m > 0)
    neg = np.array([at[(l[i], -m[i])] for i in pos], dtype=np.int64)
    return pos, neg, np.where(m[pos] & 1, -1.0, 1.0)


def _coeffs(bw, fields, real, seed, dev):
    """Power-law coefficients, E|c|^2 = (l+1)^-2; for real data the coefficients of real fields."""
    re, im = synth.power_law_coeffs(bw, fields, seed, dev)
    if real:
        pos, neg, sg = _neg_rows(bw)
        pos, neg = torch.tensor(pos, device=dev), torch.tensor(neg, device=dev)
        sg = torch.tensor(sg, dtype=torch.float64, device=dev)
        re[:, neg] = re[:, pos] * sg
        im[:, neg] = -im[:, pos] * sg
        im[:, :bw] = 0
    return re, im


def _filters(bw, fields, seed, dev):
    """Gaussian filters on the grid, constant along phi, of widths drawn per filter."""
    n = 2 * bw
    rng = np.random.default_rng(seed)
    s = torch.tensor(rng.uniform(2.0 / bw, 0.4, fields), dtype=torch.float64, device=dev)
    th = (2 * torch.arange(n, dtype=torch.float64, device=dev) + 1) * (math.pi / (2 * n))
    h = torch.exp(-0.5 * (th[None, :] / s[:, None]) ** 2)
    return h[:, :, None].expand(fields, n, n).contiguous()


_CONV_BWS = (32, 64, 128, 256, 512)
_CONV_P = (0.3, 0.3, 0.2, 0.15, 0.05)


def _conv_groups(case, seed):
    """Request bandwidths in request order; the counts are the same for every seed."""
    sizes = [b for b in _CONV_BWS if b <= case["bw"]]
    p = _CONV_P[:len(sizes)]
    counts = [max(1, int(case["fields"] * x / sum(p))) for x in p]
    bws = np.concatenate([np.full(c, b) for b, c in zip(sizes, counts)])
    return np.random.default_rng(seed).permutation(bws)


def _conv_inputs(case, seed, dev):
    bws = _conv_groups(case, seed)
    data = {}
    for bw in sorted(set(bws.tolist())):
        c = int((bws == bw).sum())
        sr, si = _grids(bw, c, True, seed + bw, dev)
        hr = _filters(bw, c, seed + bw, dev)
        data[bw] = (sr, si, hr, torch.zeros_like(hr))
    return bws, data


def prepare(case, seed):
    kind, bw, fields, real = case["kind"], case["bw"], case["fields"], case["real"]
    fmt = S.REAL if real else S.COMPLEX
    dev = _dev()
    if kind == "dropin_conv":
        sr, si = (t[0].cpu().numpy() for t in _grids(bw, 1, True, seed, dev))
        hr = _filters(bw, 1, seed, dev)[0].cpu().numpy()
        return {"kind": kind, "bw": bw, "in": (sr, si, hr, np.zeros_like(hr))}
    if kind == "conv_batch":
        bws, data = _conv_inputs(case, seed, dev)
        out = {b: (torch.empty_like(t[0]), torch.empty_like(t[0])) for b, t in data.items()}
        slot, reqs = {b: 0 for b in data}, []
        for b in bws.tolist():
            j = slot[b]
            slot[b] += 1
            reqs.append((b, *[t[j] for t in data[b]], *[t[j] for t in out[b]]))
        return {"kind": kind, "batch": S.ConvBatch(reqs, precision=PREC[case["prec"]]), "out": out, "in": data}
    re, im = _grids(bw, fields, real, seed, dev)
    cr, ci = _coeffs(bw, fields, real, seed + 1, dev)
    if kind == "dropin_pair":
        return {"kind": kind, "bw": bw, "fmt": fmt, "tables": S.HostTables(bw, case["cutoff"]), "w": S.weights(bw),
                "grid": (re[0].cpu().numpy(), im[0].cpu().numpy()), "coeffs": (cr[0].cpu().numpy(), ci[0].cpu().numpy())}
    plan = S.Plan(bw, fields, precision=PREC[case["prec"]], cutoff=case["cutoff"])
    return {"kind": kind, "plan": plan, "fmt": fmt, "grid": (re, im), "coeffs": (cr, ci),
            "ogrid": (torch.empty_like(re), torch.empty_like(im)), "ocoef": (torch.empty_like(cr), torch.empty_like(ci))}


def run(s):
    kind = s["kind"]
    if kind == "dropin_conv":
        return S.conv(*s["in"], s["bw"])[0]
    if kind == "dropin_pair":
        g = S.inv_fst(*s["coeffs"], s["bw"], s["tables"], data_format=s["fmt"])
        c = S.fst(*s["grid"], s["bw"], s["tables"], w=s["w"], data_format=s["fmt"])
        return {"coeffs": c, "grid": g[0] if s["fmt"] == S.REAL else g}
    if kind == "conv_batch":
        s["batch"].run()
        return {str(b): t[0] for b, t in s["out"].items()}
    s["plan"].forward(*s["grid"], *s["ocoef"], data_format=s["fmt"])
    s["plan"].inverse(*s["coeffs"], *s["ogrid"], data_format=s["fmt"])
    return {"coeffs": s["ocoef"], "grid": s["ogrid"][0] if s["fmt"] == S.REAL else s["ogrid"]}


# ---------------------------------------------------------------------------
# work: each grid and coefficient read or written once, and the tables of the
# seminaive transform once per direction; the ring FFTs and the seminaive
# Legendre sums
# ---------------------------------------------------------------------------
def _table(bw):
    return (4 * bw ** 3 + 6 * bw ** 2 - 8 * bw) / 24 + bw


def _one_way(bw, fields, prec):
    n = 2 * bw
    el = 8 if prec == "fp64" else 4
    return (fields * 16 * (n * n + bw * bw) + el * _table(bw),
            fields * (5 * n * n * math.log2(n) + 8 * _table(bw)))


def work(case):
    if case["kind"] in ("plan", "dropin_pair"):
        b, f = _one_way(case["bw"], case["fields"], case["prec"])
        return {"bytes": 2 * b, "flops": 2 * f}
    groups = [case["bw"]] if case["kind"] == "dropin_conv" else _conv_groups(case, 0).tolist()
    b = f = 0.0
    for bw in groups:  # signal and filter grids in, output grid out
        n = 2 * bw
        b += 3 * 16 * n * n
        f += 2 * (5 * n * n * math.log2(n) + 8 * _table(bw)) + 2 * n * n
    for bw in sorted(set(groups)):
        b += 2 * (8 if case["prec"] == "fp64" else 4) * _table(bw)
    return {"bytes": b, "flops": f}


# ---------------------------------------------------------------------------
# exact: the transforms from their definitions in 64 bits
# ---------------------------------------------------------------------------
def _legendre(bw, dev):
    """T[m][l - m][j] = P_l^m(cos theta_j), L2-normalised on [-1, 1], sign (-1)^m, theta_j = (2j+1) pi/(4bw)."""
    n = 2 * bw
    th = (2 * torch.arange(n, dtype=torch.float64, device=dev) + 1) * (math.pi / (2 * n))
    x, s = torch.cos(th), torch.sin(th)
    m = torch.arange(bw, dtype=torch.float64, device=dev)[:, None]
    # P_m^m = sqrt((2m+1)!! / (2 (2m)!!)) sin^m
    k = torch.arange(1, bw, dtype=torch.float64, device=dev)
    lead = torch.cat([torch.zeros(1, dtype=torch.float64, device=dev), torch.cumsum(torch.log1p(1 / (2 * k)), 0)])
    sign = 1.0 - 2.0 * (m % 2)
    prev = torch.zeros((bw, n), dtype=torch.float64, device=dev)
    cur = sign * torch.exp(0.5 * lead[:, None] + m * torch.log(s)[None, :]) * math.sqrt(0.5)
    rows = [cur]
    for d in range(1, bw):  # l = m + d for every m at once
        l = m + d
        a = torch.sqrt((4 * l * l - 1) / (l * l - m * m))
        b = torch.sqrt(((l - 1) ** 2 - m * m) / (4 * (l - 1) ** 2 - 1))
        cur, prev = a * (x * cur - b * prev), cur
        rows.append(cur)
        if d > 1:
            rows[d - 1] = rows[d - 1][:bw - d + 1]
    return rows  # rows[d][m], m < bw - d


def _order(rows, m, bw):
    return torch.stack([rows[d][m] for d in range(bw - m)])


def _dh_weights(bw, dev):
    n = 2 * bw
    th = (2 * torch.arange(n, dtype=torch.float64, device=dev) + 1) * (math.pi / (2 * n))
    k = 2 * torch.arange(bw, dtype=torch.float64, device=dev) + 1
    return 2.0 / bw * torch.sin(th) * (torch.sin(th[:, None] * k[None, :]) / k[None, :]).sum(1)


def _slots(bw):
    """Start of order m's run of coefficients, for m and -m."""
    first = {}
    for i, m in enumerate(synth.orders(bw).tolist()):
        first.setdefault(m, i)
    return first


def _exact_forward(rows, bw, re, im, real):
    n, fields, dev = 2 * bw, re.shape[0], re.device
    w = _dh_weights(bw, dev) * (math.sqrt(2 * math.pi) / n)
    cr = torch.empty((fields, bw * bw), dtype=torch.float64, device=dev)
    ci = torch.empty_like(cr)
    ft = torch.empty((fields, n, n), dtype=torch.complex128, device=dev)
    for f in range(0, fields, 128):
        ft[f:f + 128] = torch.fft.fft(torch.complex(re[f:f + 128], im[f:f + 128]), dim=2)
    at = _slots(bw)
    for m in range(bw):
        t = (_order(rows, m, bw) * w).T.contiguous()
        for k in ((m, -m) if m else (0,)):
            sg = -1.0 if (k < 0 and m & 1) else 1.0
            if k < 0 and real:
                g = torch.conj_physical(ft[:, :, m])
            else:
                g = ft[:, :, k % n]
            sl = slice(at[k], at[k] + bw - m)
            cr[:, sl] = sg * (g.real.contiguous() @ t)
            ci[:, sl] = sg * (g.imag.contiguous() @ t)
    return cr, ci


def _exact_inverse(rows, bw, cr, ci, real):
    n, fields, dev = 2 * bw, cr.shape[0], cr.device
    ft = torch.zeros((fields, n, n), dtype=torch.complex128, device=dev)
    at = _slots(bw)
    for m in range(bw):
        t = _order(rows, m, bw) / math.sqrt(2 * math.pi)
        for k in ((m, -m) if m else (0,)):
            if k < 0 and real:
                ft[:, :, k % n] = torch.conj_physical(ft[:, :, m])
                continue
            sg = -1.0 if (k < 0 and m & 1) else 1.0
            sl = slice(at[k], at[k] + bw - m)
            ft[:, :, k % n] = sg * torch.complex(cr[:, sl].contiguous() @ t, ci[:, sl].contiguous() @ t)
    re, im = (torch.empty((fields, n, n), dtype=torch.float64, device=dev) for _ in range(2))
    for f in range(0, fields, 128):
        z = torch.fft.ifft(ft[f:f + 128], dim=2, norm="forward")
        re[f:f + 128], im[f:f + 128] = z.real, z.imag
    return re, im


def _exact_conv(bw, sr, si, hr, hi):
    rows = _legendre(bw, sr.device)
    cr, ci = _exact_forward(rows, bw, sr, si, True)
    # zonal filter: its order-0 coefficients (of a real field)
    w = _dh_weights(bw, sr.device) * (math.sqrt(2 * math.pi) / (2 * bw))
    h = (hr.sum(2) * w) @ _order(rows, 0, bw).T
    l = torch.tensor(synth.degrees(bw), device=sr.device)
    sc = torch.sqrt(4 * math.pi / (2 * l.double() + 1)) * h[:, l]
    return _exact_inverse(rows, bw, cr * sc, ci * sc, True)


def exact(case, seed):
    kind, bw, fields, real = case["kind"], case["bw"], case["fields"], case["real"]
    dev = _dev()
    # The seminaive synthesis of an odd bandwidth keeps S2kit's short rows at
    # degree bw - 1 (Transpose_RowSize): no value from the definition there.
    short = bw % 2 == 1 and case["prec"] == "fp64" and case["cutoff"] > 0
    if kind == "dropin_conv":
        if short:
            return None
        sr, si = _grids(bw, 1, True, seed, dev)
        hr = _filters(bw, 1, seed, dev)
        return _exact_conv(bw, sr, si, hr, torch.zeros_like(hr))[0].reshape(-1)
    if kind == "conv_batch":
        _, data = _conv_inputs(case, seed, dev)
        return {str(b): _exact_conv(b, *t)[0] for b, t in data.items()}
    re, im = _grids(bw, fields, real, seed, dev)
    cr, ci = _coeffs(bw, fields, real, seed + 1, dev)
    rows = _legendre(bw, dev)
    c = _exact_forward(rows, bw, re, im, real)
    g = (None, None) if short else _exact_inverse(rows, bw, cr, ci, real)
    if kind == "dropin_pair":
        c = tuple(t.reshape(-1) for t in c)
        g = tuple(t if t is None else t.reshape(-1) for t in g)
    return {"coeffs": c, "grid": g[0] if real else g}
