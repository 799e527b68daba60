"""Timed cases of the acquisition engine: what a receiver, a signal monitor or a
post-processing program asks of it, through `plan_acquire`, `acquire_` and
`acquire_batch`.

A case names a system, a sampling rate and the arguments of `plan_acquire` and
`acquire_`. `prepare` makes the samples from the seed (a few present emitters in
white noise, quantised to the case's sample type) and the plan, which such
programs keep; `run` is one search and the results it returns. `exact` is the
same search in 64 bits, written from the search's definition with torch alone.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "acquisition.jl_amd"))

from acquisition import GPSL1CA, acquire_, acquire_batch, plan_acquire  # noqa: E402
from acquisition.acquire import Packed2BitSignal  # noqa: E402
from acquisition.device import DeviceArray  # noqa: E402
from acquisition.systems import E1Like, L5Like  # noqa: E402

DEV = "cuda"
BYTES = {"cf32": 8, "cf64": 16, "i16": 2, "ci8": 2, "ci16": 4, "f32": 4, "c2bit": 0.5}
_systems = {}


def _system(name):
    if name not in _systems:
        _systems[name] = {"l1ca": GPSL1CA, "l5": L5Like, "e1": E1Like}[name]()
    return _systems[name]


def _case(system, fs, prns, *, coh=1, nnc=1, edges=1, cov=7000.0, samples="cf32", if_hz=0.0, present=1, cn0=44.0,
          precision="fp32", interp=False, host=False, surfaces=False, requests=1, **kw):
    c = dict(system=system, fs=float(fs), prns=prns, coh=coh, nnc=nnc, edges=edges, cov=float(cov), samples=samples,
             if_hz=float(if_hz), present=present, cn0=float(cn0), precision=precision, interp=interp, host=host,
             surfaces=surfaces, requests=requests)
    c.update(kw)
    return c


def listed():
    return [
        # the smallest search: a hot-start check of one satellite in 1 ms of samples
        _case("l1ca", 2.048e6, 1, name="l1ca_2mhz_1ms_1prn"),
        # cold start of a low-rate receiver, all satellites in 1 ms: launches and latency
        _case("l1ca", 5e6, 32, name="l1ca_5mhz_1ms_32prn"),
        # samples that arrive in host memory from a front end, an odd sample count per code, a few ms
        _case("l1ca", 5.115e6, 12, coh=4, nnc=3, samples="ci16", host=True, interp=True,
              name="l1ca_5115khz_4ms_x3_12prn_host"),
        # a plot of the correlation surface of a few satellites
        _case("l1ca", 4e6, 4, coh=2, surfaces=True, name="l1ca_4mhz_2ms_surfaces"),
        # assisted search of eight satellites at an SDR's rate, interpolated
        _case("l1ca", 10e6, 8, coh=5, nnc=4, cov=5000.0, samples="ci8", interp=True, name="l1ca_10mhz_5ms_x4_8prn"),
        # weak-signal search over 80 ms of real IF samples, 10 bit-edge offsets (the benchmark's search)
        _case("l1ca", 16.368e6, 32, coh=10, nnc=8, edges=10, samples="i16", if_hz=4.092e6, present=8, cn0=38.0,
              name="l1ca_16mhz_80ms_32prn"),
        # the same on a shorter 2-bit recording, half the satellites
        _case("l1ca", 16.368e6, 16, coh=10, nnc=4, edges=10, samples="c2bit", if_hz=4.092e6, present=4, cn0=40.0,
              name="l1ca_16mhz_40ms_2bit_16prn"),
        # data-bit search: two 20 ms bits, two bit-edge offsets
        _case("l1ca", 4e6, 8, coh=40, nnc=1, edges=2, present=3, name="l1ca_4mhz_40ms_databits"),
        # pilot acquisition at the wide-band rate, one code period at a time
        _case("l5", 30.69e6, 12, nnc=8, cov=5000.0, present=3, name="l5_30mhz_1ms_x8_12prn"),
        # the same over one secondary-code period: the rotation search and the secondary phase of what is found
        _case("l5", 30.69e6, 6, coh=10, nnc=2, cov=5000.0, present=2, interp=True, name="l5_30mhz_10ms_x2_6prn"),
        # BOC pilot with a 25-chip secondary code over 4 x 100 ms, default coverage
        _case("e1", 25e6, 1, coh=25, nnc=4, cov=7000.0, present=1, cn0=36.0, interp=True, name="e1_25mhz_100ms_x4"),
        # requests of several receivers in one submission
        _case("l1ca", 5e6, 8, coh=1, nnc=4, cov=10000.0, present=2, interp=True, requests=4, name="mixed_batch_4"),
    ]


# Samples per 1 ms code that front ends use: multiples of the chip rate, of 1 MHz, powers of two, odd ones.
_L1_RATES = (2046, 2048, 2500, 3069, 3125, 3375, 4000, 4092, 5000, 5115, 5250, 5456, 6138, 6144, 6500, 8000, 8184, 9000,
             10000, 10230, 12000, 12500, 15000, 16000, 16368, 16384, 20000, 20460, 25000)


def draw(rng):
    while True:
        u = rng.random()
        if u < 0.62:
            fs = rng.choice(_L1_RATES) * 1e3
            coh = rng.choice((1, 1, 2, 3, 4, 5, 8, 10, 10, 20))
            samples = rng.choice(("cf32", "cf32", "i16", "ci8", "ci16", "c2bit", "f32"))
            real = samples in ("i16", "f32")
            c = _case("l1ca", fs, int(round(math.exp(rng.uniform(0, math.log(32))))), coh=coh,
                      nnc=int(round(math.exp(rng.uniform(0, math.log(8))))), edges=rng.choice((1, coh if coh > 1 else 1)),
                      cov=rng.choice((5000.0, 7000.0, 7000.0, 10000.0)), samples=samples,
                      if_hz=fs / 4 if real else rng.choice((0.0, 0.0, 38400.0)), present=1, interp=rng.random() < 0.5,
                      host=rng.random() < 0.2)
        elif u < 0.72:
            c = _case("l1ca", rng.choice((2.048e6, 4e6, 4.092e6, 5e6)), rng.randint(1, 8), coh=40,
                      nnc=rng.choice((1, 1, 2)), edges=rng.choice((1, 2, 4)), present=1)
        elif u < 0.90:
            coh = rng.choice((1, 1, 10))
            c = _case("l5", 30.69e6, rng.randint(1, 16), coh=coh, nnc=rng.randint(1, 4), cov=rng.choice((5000.0, 10000.0)),
                      present=1, interp=rng.random() < 0.5)
        else:
            c = _case("e1", 25e6, 1, coh=25, nnc=rng.choice((1, 2)), cov=rng.choice((5000.0, 7000.0, 10000.0, 25000.0)),
                      present=rng.choice((0, 1)), interp=True, precision=rng.choice(("fp32", "auto")))
        if c["edges"] > 1 and c["coh"] < 20 and c["coh"] % c["edges"]:
            continue
        g = _geometry(c)
        if g["ndop"] > 4000 and c["system"] == "l1ca":
            continue  # a rate with no suitable block count
        big = _geometry(listed()[-2])
        if _cells(c, g) <= _cells(listed()[-2], big):
            return c


# ---------------------------------------------------------------------------
# geometry of a search (the definition of plan_acquire)
# ---------------------------------------------------------------------------
def _geometry(c):
    s = _system(c["system"])
    spc = math.ceil(s.code_length / s.code_frequency * c["fs"])
    lo = math.ceil(2 * c["cov"] / (c["fs"] / spc) + 2 / c["coh"])
    nb = next(b for b in range(max(lo, 1), spc + 1) if spc % b == 0)
    L = s.get_secondary_code_length()
    rot = L if L > 1 and c["coh"] > 1 else 1
    bits = 1
    if c["system"] == "l1ca" and c["coh"] >= 20:
        bits = c["coh"] // 20
    return dict(spc=spc, nb=nb, bs=spc // nb, ndop=c["coh"] * nb, R=rot, ndb=bits, n=spc * c["coh"] * c["nnc"])


def _cells(c, g):
    return c["requests"] * c["prns"] * g["ndop"] * g["spc"] * g["R"] * c["nnc"]


def work(case):
    g = _geometry(case)
    fft = 5.0 * g["spc"] * math.log2(g["spc"])
    # one circular correlation of the code period per Doppler bin, rotation and step
    flops = case["requests"] * case["prns"] * case["nnc"] * g["ndop"] * g["R"] * (fft + 10.0 * g["spc"])
    nbytes = case["requests"] * (g["n"] * BYTES[case["samples"]] + case["prns"] * (g["spc"] + 64))
    if case["surfaces"]:
        nbytes += 4.0 * case["prns"] * g["ndop"] * g["spc"] * g["R"]
    return {"bytes": float(nbytes), "flops": float(flops)}


# ---------------------------------------------------------------------------
# samples
# ---------------------------------------------------------------------------
def _samples(c, g, seed):
    """Complex or real samples of the case as a float64 / complex128 tensor in
    the units of its sample type, already quantised."""
    s = _system(c["system"])
    gen = torch.Generator(device=DEV).manual_seed(seed)
    host = torch.Generator().manual_seed(seed)
    n, fs = g["n"], c["fs"]
    t = torch.arange(n, dtype=torch.float64, device=DEV)
    real = c["samples"] in ("i16", "f32")
    scale = {"i16": 1000.0, "ci8": 32.0, "ci16": 500.0}.get(c["samples"], 1.0)
    if real:
        x = torch.randn(n, generator=gen, dtype=torch.float64, device=DEV)
    else:
        x = torch.complex(torch.randn(n, generator=gen, dtype=torch.float64, device=DEV),
                          torch.randn(n, generator=gen, dtype=torch.float64, device=DEV)) / math.sqrt(2.0)
    sec = torch.as_tensor(s.secondary_code(1).astype(np.float64), device=DEV)
    for e in range(c["present"]):
        prn = 1 + e * max(1, c["prns"] // max(1, c["present"]))
        u = torch.rand(5, generator=host, dtype=torch.float64).tolist()
        fd = (2 * u[0] - 1) * 0.8 * min(c["cov"], 5000.0)
        chips = torch.as_tensor(s.primary_chips(prn).astype(np.float64), device=DEV)
        pos = u[1] * s.code_length + t * ((s.code_frequency + fd * s.code_frequency / s.center_frequency) / fs)
        whole = torch.floor(pos)
        idx = whole.to(torch.int64)
        a = chips[idx % s.code_length]
        if s.boc:
            a = torch.where(pos - whole < 0.5, a, -a)
        if len(sec) > 1:
            a = a * sec[(idx // s.code_length + int(u[4] * len(sec))) % len(sec)]
        if c["system"] == "l1ca":
            bit = torch.randint(0, 2, (n // int(fs // 50) + 3,), generator=host).to(DEV).double() * 2 - 1
            a = a * bit[((t * (1000.0 / fs)).floor().to(torch.int64) + int(u[4] * 20)) // 20]
        ph = 2 * math.pi * (torch.remainder(t * ((c["if_hz"] + fd) / fs), 1.0) + u[2])
        amp = 10 ** ((c["cn0"] + 3 * u[3]) / 20) / math.sqrt(fs)
        x = x + (2 * amp * a * torch.cos(ph) if real else amp * a * torch.exp(1j * ph))
    x = x * scale
    if c["samples"] == "i16":
        return x.round().clamp(-32768, 32767)
    if c["samples"] == "f32":
        return x.float().double()
    if c["samples"] == "cf32":
        return x.to(torch.complex64).to(torch.complex128)
    if c["samples"] == "c2bit":
        def level(v):
            return torch.where(v >= 0, 1.0, -1.0) * torch.where(v.abs() >= math.sqrt(0.5), 3.0, 1.0)

        return torch.complex(level(x.real).double(), level(x.imag).double())
    top = 127 if c["samples"] == "ci8" else 32767
    return torch.complex(x.real.round().clamp(-top, top), x.imag.round().clamp(-top, top))


def _as_signal(c, x):
    """The samples as a program holds them: in device memory, or host arrays."""
    k = c["samples"]
    if k == "cf32":
        y = x.to(torch.complex64)
    elif k in ("i16", "f32"):
        y = x.to(torch.int16 if k == "i16" else torch.float32)
    elif k in ("ci8", "ci16"):
        y = torch.view_as_real(x).to(torch.int8 if k == "ci8" else torch.int16).contiguous()
    else:
        p = Packed2BitSignal.pack(torch.view_as_real(x).cpu().numpy())
        return p if c["host"] else Packed2BitSignal(DeviceArray(p.packed), p.n)
    return y.cpu().numpy() if c["host"] else y


def _kinds(case):
    """The requests of a case: itself, or the several of a batch."""
    if case["requests"] == 1:
        return [case]
    out = []
    for i in range(case["requests"]):
        k = dict(case, requests=1)
        if i % 4 == 1:
            k.update(fs=4e6, coh=2, nnc=2, prns=max(1, case["prns"] // 2))
        elif i % 4 == 2:
            k.update(fs=8.184e6, coh=5, nnc=1, cov=5000.0, samples="ci8")
        elif i % 4 == 3:
            k.update(system="l5", fs=30.69e6, coh=1, nnc=2, cov=5000.0, prns=max(1, case["prns"] // 4), present=1)
        out.append(k)
    return out


def prepare(case, seed):
    reqs = []
    for i, c in enumerate(_kinds(case)):
        prns = list(range(1, c["prns"] + 1))
        signal = _as_signal(c, _samples(c, _geometry(c), seed + 7919 * i))
        plan = plan_acquire(_system(c["system"]), c["fs"], prns, min_doppler_coverage=c["cov"],
                            num_coherently_integrated_code_periods=c["coh"], bit_edge_search_steps=c["edges"],
                            num_noncoherent_accumulations=c["nnc"], tile_precision=c["precision"])
        kw = dict(interm_freq=c["if_hz"], subsample_interpolation=c["interp"], store_power_bins=c["surfaces"])
        reqs.append((plan, signal, prns, kw))
    return reqs


def _outputs(results, interp):
    place, cn0, noise, ptn, sec = zip(*[((r.code_phase, r.carrier_doppler), r.CN0, r.noise_power, r.peak_to_noise_ratio,
                                         -1 if r.secondary_code_phase is None else r.secondary_code_phase)
                                        for r in results])
    # positions on the search grid are exact; interpolated ones and powers are 32-bit results
    return {"place": np.array(place, dtype=np.float32 if interp else np.float64),
            "cn0": np.array(cn0, dtype=np.float32), "noise": np.array(noise, dtype=np.float32),
            "ptn": np.array(ptn, dtype=np.float32), "secondary": np.array(sec, dtype=np.int64)}


def run(state):
    if len(state) > 1:
        found = acquire_batch(state)
        return [_outputs(r, kw["subsample_interpolation"]) for r, (_, _, _, kw) in zip(found, state)]
    plan, signal, prns, kw = state[0]
    found = acquire_(plan, signal, prns, **kw)
    out = _outputs(found, kw["subsample_interpolation"])
    if kw["store_power_bins"]:
        out["surfaces"] = [r.power_bins for r in found]
    return out


# ---------------------------------------------------------------------------
# the search in 64 bits
# ---------------------------------------------------------------------------
def exact(case, seed):
    out = [_exact_request(c, seed + 7919 * i) for i, c in enumerate(_kinds(case))]
    if any(o is None for o in out):
        return None
    return out if len(out) > 1 else out[0]


def _mixed(c, g, x):
    """Samples at baseband. The search's carrier phase is defined on Float32
    values (step and products rounded to Float32); everything after is 64 bits."""
    if c["if_hz"] == 0.0:
        return x.to(torch.complex128)
    f = np.float32
    step = f(-2 * math.pi * c["if_hz"] / c["fs"])
    seg = g["spc"] * c["coh"]
    ph = np.concatenate([(f(f(m * seg) * step) + np.arange(seg).astype(f) * step).astype(f) for m in range(c["nnc"])])
    return x * torch.exp(1j * torch.as_tensor(ph.astype(np.float64), device=DEV))


def _code(s, prn, g, fs):
    pos = np.arange(g["spc"], dtype=np.float64) * s.code_frequency / fs
    k = np.floor(pos).astype(np.int64)
    a = s.primary_chips(prn)[k % s.code_length].astype(np.float64)
    if s.boc:
        a = np.where(pos - np.floor(pos) < 0.5, a, -a)
    return torch.as_tensor(a, device=DEV)


def _tile(g, z, code):
    """tile[k][r * bs + lag]: the correlation of double block k of one segment
    with code block (k + r) mod nb."""
    nb, bs, ndop = g["nb"], g["bs"], g["ndop"]
    F = 2 * bs
    zz = torch.cat([z, z[:bs]]).unfold(0, F, bs)
    S = torch.fft.fft(zz, dim=1)
    P = torch.fft.fft(code.to(torch.complex128).view(nb, bs), n=F, dim=1).conj()
    out = torch.empty((ndop, nb, bs), dtype=torch.complex128, device=DEV)
    k = torch.arange(ndop, device=DEV)
    for r in range(nb):
        out[:, r] = torch.fft.ifft(S * P[(k + r) % nb], dim=1)[:, :bs]
    return out.view(ndop, nb * bs)


def _column_powers(c, g, tile, c0, c1, sec):
    """Power surfaces [R][rows, sorted Doppler][columns c0..c1) of one segment."""
    ndop, nb, bs, coh = g["ndop"], g["nb"], g["bs"], c["coh"]
    half = ndop // 2
    x = tile[:, c0:c1]
    if g["R"] > 1:
        cp = torch.arange(c0, c1, device=DEV)
        wrap = ((nb - cp // bs) % nb) * bs + cp % bs
        eff = ((wrap + bs // 2) // bs) % nb
        rows = (torch.arange(ndop, device=DEV)[:, None] + eff[None, :]) % ndop
        x = torch.gather(x, 0, rows)
        out = []
        for q in range(g["R"]):
            sg = torch.as_tensor([float(sec[(p + q) % len(sec)]) for p in range(coh)], device=DEV, dtype=torch.float64)
            y = torch.fft.fft(x * sg.repeat_interleave(nb)[:, None], dim=0)
            out.append(torch.roll(y.real.square() + y.imag.square(), half, 0))
        return torch.stack(out)
    if g["ndb"] == 1:
        y = torch.fft.fft(x, dim=0)  # every bit-edge offset has the same power
        return torch.roll(y.real.square() + y.imag.square(), half, 0)[None]
    sub = ndop // g["ndb"]
    edge = (coh // g["ndb"]) * nb // c["edges"]
    best = None
    for e in range(c["edges"]):
        b = torch.roll(x, -e * edge, 0).view(g["ndb"], sub, c1 - c0)
        for d in range(1 << (g["ndb"] - 1)):
            y = b[0]
            for i in range(1, g["ndb"]):
                y = y + (-1.0 if (d >> (i - 1)) & 1 else 1.0) * b[i]
            y = torch.fft.fft(y, n=ndop, dim=0)
            y = torch.roll(y.real.square() + y.imag.square(), half, 0)
            best = y if best is None else torch.maximum(best, y)
    return best[None]


def _exact_request(c, seed):
    g = _geometry(c)
    s = _system(c["system"])
    spc, ndop, R = g["spc"], g["ndop"], g["R"]
    if 8.0 * R * ndop * spc > 60e9 or _cells(c, g) > 2.5e10:
        return None  # over about 20 seconds
    z = _mixed(c, g, _samples(c, g, seed)).view(c["nnc"], -1)
    spacing = (c["fs"] / spc) / c["coh"]
    doppler = np.array([-g["nb"] * c["fs"] / spc / 2 + i * spacing for i in range(ndop)])
    place, cn0, noise, ptn, surfaces = [], [], [], [], []
    chunk = max(1, min(spc, int(2e9 // (16 * ndop * 4))))
    for prn in range(1, c["prns"] + 1):
        code, sec = _code(s, prn, g, c["fs"]), s.secondary_code(prn)
        acc = torch.zeros((R, ndop, spc), dtype=torch.float64, device=DEV)
        for m in range(c["nnc"]):
            tile = _tile(g, z[m], code)
            shift = torch.as_tensor([round(f * m * (c["coh"] * spc / c["fs"]) * c["fs"] / s.center_frequency) % spc
                                     for f in doppler.tolist()], device=DEV)
            for c0 in range(0, spc, chunk):
                c1 = min(spc, c0 + chunk)
                pw = _column_powers(c, g, tile, c0, c1, sec)
                to = (torch.arange(c0, c1, device=DEV)[None, :] + shift[:, None]) % spc
                for q in range(R):
                    acc[q].scatter_add_(1, to, pw[q])
            del tile
        at = int(acc.view(-1).argmax())
        q, row, col = at // (ndop * spc), at // spc % ndop, at % spc
        peak = acc[q, row, col].item()
        nz = acc[:, (row + ndop // 2) % ndop].mean().item()
        delay = ((g["nb"] - col // g["bs"]) % g["nb"]) * g["bs"] + col % g["bs"]
        d, fd = float(delay), float(doppler[row])
        if c["interp"]:
            a, b = acc[q, row, (col - 1) % spc].item(), acc[q, row, (col + 1) % spc].item()
            if max(a, b) > math.sqrt(nz):
                d += (b - a) / (2 * (2 * peak - a - b))
            a, b = acc[q, (row - 1) % ndop, col].item(), acc[q, (row + 1) % ndop, col].item()
            if max(a, b) > math.sqrt(nz):
                fd += (b - a) / (2 * (2 * peak - a - b)) * spacing
        place.append((math.fmod(-d * s.code_frequency / c["fs"], s.code_length) % s.code_length, fd))
        cn0.append(10 * math.log10((peak - nz) / nz / (c["coh"] * s.code_length / s.code_frequency)))
        noise.append(nz)
        ptn.append(peak / nz)
        if c["surfaces"]:
            surfaces.append(acc.permute(1, 0, 2).reshape(ndop, R * spc))
        del acc
    out = {"place": np.array(place), "cn0": np.array(cn0), "noise": np.array(noise), "ptn": np.array(ptn),
           "secondary": None}
    if c["surfaces"]:
        out["surfaces"] = surfaces
    return out
