"""The calls that programs built on qstem_amd spend their time in, as measurable cases.

Every case goes through the public entry points (Multislice, run_groups, multislice_loss)
and is a dict of plain values; `kind` says what it stands for:

  scan    a STEM scan: probe positions through a specimen, detector images back
  wave    one plane or probe wave through a specimen, its exit wave back (TEM, CBED)
  groups  windows of several sizes over shared frozen-phonon configurations
  probes  gradients of a 4D-STEM diffraction loss (potential, defocus, Cs)
  image   gradients of the same loss for one plane wave over the whole grid
  atoms   one frozen-phonon run from atom positions: potential, probe, scan

Inputs are made on the GPU from the seed: projected potentials of randomly placed atoms
(Gaussian columns of 3 to 30 V A^2 peak, about one per 12 A^2 and slice).  exact() computes
the same outputs in 64 bits with plain torch.
"""
import math

import numpy as np
import torch

from qstem_amd import Detector, Multislice, StemConfig, record_bins, run_groups
from qstem_amd.autograd import multislice_loss

DETECTORS = ((0.0, 10.0), (11.0, 22.0), (40.0, 100.0))  # bright field, annular bright field, annular dark field (mrad)
CELL = 3.905  # perovskite cell edge of the atom models (A)
# Sr, Ti, O as in the SrTiO3 model of the tests: fractional position, Z, Debye-Waller factor, charge
BASIS = ((0.0, 0.0, 0.0, 38, 0.6214, 2.0), (0.5, 0.5, 0.5, 22, 0.4390, 4.0), (0.0, 0.5, 0.5, 8, 0.7323, -2.0),
         (0.5, 0.0, 0.5, 8, 0.7323, -2.0), (0.5, 0.5, 0.0, 8, 0.7323, -2.0))
RADIUS = 5.0  # atom radius of the potential (A)


def listed():
    return [
        # one probe position, looked at by itself: launches and host time, hardly any arithmetic
        dict(name="probe_128", kind="scan", nx=128, ny=128, pad=97, dx=0.040, kv=200.0, slices=20, probes=1, every=0,
             configs=1, limit=1),
        # the small scan of the benchmark's CPU configuration
        dict(name="scan_128", kind="scan", nx=128, ny=128, pad=97, dx=0.040, kv=200.0, slices=20, probes=256, every=0,
             configs=1, limit=1),
        # a short line scan at the headline size: far fewer probes than fill the GPU well
        dict(name="line_512", kind="scan", nx=512, ny=512, pad=130, dx=0.030, kv=300.0, slices=40, probes=17, every=0,
             configs=1, limit=1),
        # the headline workload's window and potential grid: a call of its 64 x 64 scan (half the
        # thickness, twice the positions: the detector sums' single-precision error grows with the
        # slices, and at 80 it is as large as the differences that are to be told apart)
        dict(name="scan_512", kind="scan", nx=512, ny=512, pad=130, dx=0.030, kv=300.0, slices=40, probes=512, every=0,
             configs=1, limit=1),
        # the 20 x 20 scan of stem_STO_4x4.qsc: no power of two, images every 8 slices, no transmission band limit
        dict(name="scan_400", kind="scan", nx=400, ny=400, pad=128, dx=0.0625, kv=200.0, slices=40, probes=400, every=8,
             configs=1, limit=0),
        # a rectangular window of lengths without compiled plans
        dict(name="scan_480x336", kind="scan", nx=480, ny=336, pad=61, dx=0.050, kv=200.0, slices=30, probes=101,
             every=10, configs=1, limit=1),
        # large windows over two phonon configurations
        dict(name="scan_1024", kind="scan", nx=1024, ny=1024, pad=64, dx=0.080, kv=200.0, slices=32, probes=48, every=0,
             configs=2, limit=1),
        # plane-wave TEM image simulation
        dict(name="wave_4096", kind="wave", n=4096, dx=0.0953, kv=300.0, slices=60, limit=1),
        # mixed window sizes over shared phonon configurations (6 : 4 : 2 positions per configuration)
        dict(name="groups_1088", kind="groups", pot=1088, small=256, dx=0.080, kv=200.0, slices=30, configs=8, each=1),
        # 4D-STEM reconstruction step: 32 x 32 positions
        dict(name="probes_256", kind="probes", n=256, pad=128, dx=0.050, kv=200.0, slices=20, probes=1024, limit=1),
        # gradient of one large image
        dict(name="image_4096", kind="image", n=4096, dx=0.0953, kv=300.0, slices=24, limit=1),
        # one frozen-phonon run of stem_STO_4x4.qsc: potential of 8100 charged atoms, probe, scan
        dict(name="atoms_400", kind="atoms", n=400, pad=128, dx=0.0625, kv=200.0, slices=40, cells=9, probes=400,
             every=8),
    ]


POWERS = (64, 128, 256, 512, 1024, 2048, 4096)
MOST = 512 * 40 * 512 * 512  # probe-slice pixels of the largest scan


def _spread(rng, lo, hi):
    """A whole number from lo to hi, spread over its logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1)))))))


def _window(rng):
    """A wave grid: powers of two, lengths of small prime factors, and now and then any length."""
    what = rng.random()
    if what < 0.55:
        nx = rng.choice(POWERS[:5])
        return nx, (nx if rng.random() < 0.7 else rng.choice(POWERS[:5]))
    if what < 0.9:
        smooth = [n for n in range(96, 641, 2) if max(_factors(n)) <= 7 and n & (n - 1)]
        nx = rng.choice(smooth)
        return nx, (nx if rng.random() < 0.7 else rng.choice(smooth))
    nx = rng.randrange(80, 420)
    return nx, nx


def _factors(n):
    f, p = [], 2
    while n > 1:
        while n % p == 0:
            f.append(p)
            n //= p
        p += 1
    return f


def draw(rng):
    kind = rng.choice(("scan", "scan", "scan", "scan", "wave", "groups", "probes", "image", "atoms"))
    if kind == "scan":
        nx, ny = _window(rng)
        slices = _spread(rng, 4, 48)
        # lengths with a prime factor above 7 take several times as long for each pixel
        most = MOST // (16 if max(_factors(nx) + _factors(ny)) > 7 else 1)
        probes = _spread(rng, 1, max(1, min(700, most // (slices * nx * ny))))
        return dict(kind=kind, nx=nx, ny=ny, pad=rng.randrange(3, 161), dx=rng.uniform(0.03, 0.08),
                    kv=rng.choice((100.0, 200.0, 300.0)), slices=slices, probes=probes,
                    every=rng.choice((0, 0, max(1, slices // 4))), configs=rng.choice((1, 1, 2)),
                    limit=rng.choice((1, 1, 0)))
    if kind == "wave":
        n = rng.choice(POWERS[2:])
        return dict(kind=kind, n=n, dx=rng.uniform(0.05, 0.1), kv=rng.choice((200.0, 300.0)),
                    slices=_spread(rng, 8, 60), limit=rng.choice((1, 1, 0)))
    if kind == "groups":
        return dict(kind=kind, pot=rng.randrange(1030, 1160), small=rng.choice((128, 256)), dx=rng.uniform(0.05, 0.08),
                    kv=200.0, slices=_spread(rng, 6, 30), configs=rng.randrange(2, 9), each=1)
    if kind == "probes":
        n = rng.choice(POWERS[:4])
        slices = _spread(rng, 4, 20)
        probes = _spread(rng, 2, max(4, min(1500, 20 * 1024 * 65536 // (slices * n * n))))
        return dict(kind=kind, n=n, pad=rng.randrange(16, 150), dx=rng.uniform(0.04, 0.08), kv=rng.choice((100.0, 200.0)),
                    slices=slices, probes=probes, limit=rng.choice((1, 0)))
    if kind == "image":
        return dict(kind=kind, n=rng.choice(POWERS[3:]), dx=rng.uniform(0.06, 0.1), kv=rng.choice((200.0, 300.0)),
                    slices=_spread(rng, 4, 24), limit=rng.choice((1, 1, 0)))
    n = rng.choice((256, 300, 360, 400, 512))
    slices = 2 * rng.randrange(4, 21)
    return dict(kind=kind, n=n, pad=rng.randrange(32, 129), dx=rng.uniform(0.05, 0.0625), kv=200.0, slices=slices,
                cells=rng.randrange(6, 10), probes=_spread(rng, 4, 400), every=0)


# ---- inputs ------------------------------------------------------------------------

def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _potential(seed, slices, nx, ny, dx):
    """[slices][nx][ny] float32 on the GPU: Gaussian atom columns at random places."""
    g = _generator(seed)
    kx = torch.fft.fftfreq(nx, d=dx, device="cuda")[:, None]
    ky = torch.fft.rfftfreq(ny, d=dx, device="cuda")[None, :]
    sigma = 0.25
    shape = torch.exp(-2 * (math.pi * sigma) ** 2 * (kx ** 2 + ky ** 2)) * (2 * math.pi * sigma ** 2 / dx ** 2)
    V = torch.empty(slices, nx, ny, device="cuda")
    for s in range(slices):
        there = torch.rand(nx, ny, generator=g, device="cuda") < dx * dx / 12.0
        peak = 3.0 + 27.0 * torch.rand(nx, ny, generator=g, device="cuda")
        V[s] = torch.fft.irfft2(torch.fft.rfft2(there * peak) * shape, s=(nx, ny)).clamp_(min=0.0)
    return V


def _raster(nx, ny, pad, probes):
    """Window offsets of a raster over the whole margin, [probes][2]."""
    rows = max(1, int(math.sqrt(probes)))
    cols = -(-probes // rows)
    i = np.arange(probes)
    x = np.rint((i // cols) * (pad / max(1, rows - 1))) if rows > 1 else np.zeros(probes)
    y = np.rint((i % cols) * (pad / max(1, cols - 1))) if cols > 1 else np.zeros(probes)
    return np.stack([np.minimum(x, pad), np.minimum(y, pad)], 1).astype(np.int32)


def _config(nx, ny, potx, poty, dx, kv, slices, limit, **more):
    f = dict(nx=nx, ny=ny, resolutionX=dx, resolutionY=dx, v0=kv, slices=slices, sliceThickness=CELL / 2, potNx=potx,
             potNy=poty, bandlimittrans=limit, Cs=1.0e4, df0=-50.0, alpha=20.0, electronScale=1.0,
             detectors=[Detector(lo, hi, "detector%d" % i) for i, (lo, hi) in enumerate(DETECTORS)])
    f.update(more)
    return StemConfig(**f)


def _atoms(case, seed):
    """(n, 7) atoms of a block of perovskite cells displaced as Einstein phonons, x and y
    offsets of the potential, by z."""
    cells, layers = case["cells"], case["slices"] // 2
    rng = np.random.default_rng(seed)
    at = np.stack(np.meshgrid(np.arange(cells), np.arange(cells), np.arange(layers), indexing="ij"), -1).reshape(-1, 1, 3)
    b = np.array(BASIS)
    xyz = ((at + b[None, :, :3]) * CELL).reshape(-1, 3)
    Z, dw, q = (np.tile(b[:, k], len(at)) for k in (3, 4, 5))
    xyz = xyz + rng.standard_normal(xyz.shape) * (np.sqrt(dw / (8 * np.pi ** 2) / 3.0))[:, None]
    atoms = np.column_stack([xyz, dw, np.ones(len(xyz)), q, Z])
    middle = 0.5 * (cells * CELL - (case["n"] + case["pad"]) * case["dx"])
    return atoms[np.argsort(atoms[:, 2], kind="stable")], float(np.float32(middle))


def _group_plan(case):
    """(window, offsets, configuration of each) of the three window sizes of a `groups` case."""
    for k, n in enumerate((case["small"], 512, 1024)):
        per = (6, 4, 2)[k] * case["each"]
        g = np.rint(np.linspace(0, case["pot"] - n, per)).astype(np.int32)
        yield n, np.tile(np.stack([g, g[::-1]], 1), (case["configs"], 1)), np.repeat(np.arange(case["configs"], dtype=np.int32), per)


def prepare(case, seed):
    kind = case["kind"]
    if kind == "scan":
        nx, ny, pad = case["nx"], case["ny"], case["pad"]
        ms = Multislice(_config(nx, ny, nx + pad, ny + pad, case["dx"], case["kv"], case["slices"], case["limit"]))
        ms.set_configs(case["configs"])
        for k in range(case["configs"]):
            ms.select_config(k)
            ms.set_potential(_potential(seed * 8 + k, case["slices"], nx + pad, ny + pad, case["dx"]))
        ms.make_probe()
        bins, nbins = record_bins(case["slices"], outputInterval=case["every"])
        config = np.arange(case["probes"], dtype=np.int32) % case["configs"] if case["configs"] > 1 else None
        return dict(kind=kind, ms=ms, ipos=_raster(nx, ny, pad, case["probes"]), bins=bins, nbins=nbins, config=config)
    if kind == "groups":
        made = []
        for n, ipos, config in _group_plan(case):
            ms = Multislice(_config(n, n, case["pot"], case["pot"], case["dx"], case["kv"], case["slices"], 1))
            if not made:
                ms.set_configs(case["configs"])
                for k in range(case["configs"]):
                    ms.select_config(k)
                    ms.set_potential(_potential(seed * 8 + k, case["slices"], case["pot"], case["pot"], case["dx"]))
            else:
                ms.share_trans(made[0][0])
            ms.make_probe()
            made.append((ms, ipos, config))
        bins, nbins = record_bins(case["slices"])
        return dict(kind=kind, groups=made, bins=bins, nbins=nbins)
    if kind == "atoms":
        n, pot = case["n"], case["n"] + case["pad"]
        ms = Multislice(_config(n, n, pot, pot, case["dx"], case["kv"], case["slices"], 0))
        ms.set_scattering_table()
        ms.set_ion_scattering_table()
        atoms, offset = _atoms(case, seed)
        bins, nbins = record_bins(case["slices"], outputInterval=case["every"])
        return dict(kind=kind, ms=ms, atoms=atoms, offset=offset, ipos=_raster(n, n, case["pad"], case["probes"]),
                    bins=bins, nbins=nbins)
    n, pad = case["n"], case.get("pad", 0)
    ms = Multislice(_config(n, n, n + pad, n + pad, case["dx"], case["kv"], case["slices"], case["limit"]))
    V = _potential(seed, case["slices"], n + pad, n + pad, case["dx"])
    ipos = _raster(n, n, pad, case.get("probes", 1))
    if kind == "probes":
        leaf = lambda v: torch.tensor(v, dtype=torch.float32, requires_grad=True)  # noqa: E731
        return dict(kind=kind, ms=ms, V=V.requires_grad_(), df0=leaf(-50.0), Cs=leaf(1.0e4), ipos=ipos,
                    target=_target(case, V.detach(), ipos))
    ms.set_potential(V)
    ms.set_incident_wave(np.ones((n, n), np.complex64))
    return dict(kind=kind, ms=ms, ipos=ipos, target=_target(case, V, ipos) if kind == "image" else None)


def run(state):
    kind = state["kind"]
    if kind == "scan":
        out = state["ms"].run_stem(state["ipos"], bins=state["bins"], nbins=state["nbins"], config=state["config"],
                                   want_intensity=True)
        return {"det": out["det"], "intensity": out["intensity"]}
    if kind == "wave":
        return {"exit": state["ms"].run_stem(state["ipos"], want_det=False, want_exit=True)["exit"]}
    if kind == "groups":
        return [out["det"] for out in run_groups(state["groups"], bins=state["bins"], nbins=state["nbins"])]
    if kind == "atoms":
        ms = state["ms"]
        ms.build_potential(state["atoms"], atomRadius=RADIUS, potOffsetX=state["offset"], potOffsetY=state["offset"],
                           czOffset=CELL / 4, tds=1)
        ms.make_probe()
        return {"det": ms.run_stem(state["ipos"], bins=state["bins"], nbins=state["nbins"])["det"]}
    if kind == "probes":
        V, df0, Cs = state["V"], state["df0"], state["Cs"]
        V.grad = df0.grad = Cs.grad = None
        loss = multislice_loss(V, df0, Cs, state["ms"], state["ipos"], state["target"])
        loss.backward()
        # the library computes the loss in single precision
        return {"loss": loss.detach().float(), "V": V.grad, "df0": df0.grad, "Cs": Cs.grad}
    ms = state["ms"]
    loss = ms.forward_save(state["ipos"], state["target"])
    grad = ms.adjoint_saved(want_grad_V=True, want_grad_probe=False, device="cuda")
    return {"loss": np.float32(loss), "V": grad["grad_V"]}


def work(case):
    """Compulsory traffic (transmission functions or potentials once, outputs once) and the
    floating-point operations of the slice steps: transmit, two 2D transforms, propagate."""
    kind = case["kind"]

    def step(nx, ny):
        return nx * ny * (2 * 5 * math.log2(nx * ny) + 12)

    if kind == "scan":
        items = case["probes"] * case["slices"]
        pot = (case["nx"] + case["pad"]) * (case["ny"] + case["pad"]) * case["slices"] * case["configs"]
        return {"bytes": 8.0 * pot + 16.0 * case["probes"], "flops": items * step(case["nx"], case["ny"])}
    if kind == "wave":
        n2 = case["n"] ** 2
        return {"bytes": 8.0 * n2 * (case["slices"] + 2), "flops": case["slices"] * step(case["n"], case["n"])}
    if kind == "groups":
        return {"bytes": 8.0 * case["pot"] ** 2 * case["slices"] * case["configs"],
                "flops": case["slices"] * sum(len(ipos) * step(n, n) for n, ipos, _ in _group_plan(case))}
    if kind == "atoms":
        pot = (case["n"] + case["pad"]) ** 2 * case["slices"]
        samples = case["cells"] ** 2 * case["slices"] / 2 * len(BASIS) * math.pi * (RADIUS / case["dx"]) ** 2 * 6
        return {"bytes": 12.0 * pot, "flops": samples * 8 + case["probes"] * case["slices"] * step(case["n"], case["n"])}
    n, pad, probes = case["n"], case.get("pad", 0), case.get("probes", 1)
    # forward, and twice the forward's transforms back; V in, dL/dV out, the target in
    return {"bytes": 8.0 * (n + pad) ** 2 * case["slices"] + 4.0 * probes * n * n,
            "flops": 3 * probes * case["slices"] * step(n, n)}


# ---- the same outputs in 64 bits ------------------------------------------------------

def _wavelength(kv):
    return 12.3984244 / math.sqrt(kv * (2.0 * 510.99906 + kv))


def _k2(n, size):
    """Squared spatial frequencies in single precision, which decides what a mask keeps."""
    i = np.arange(n)
    k = np.where(i > n // 2, i - n, i).astype(np.float32) / np.float32(size)
    return torch.from_numpy(k * k).cuda()


def _band(nx, ny, sx, sy):
    """Pixels inside 2/3 of the smaller Nyquist limit, single-precision sums."""
    half = min(np.float32(nx) / (np.float32(2) * np.float32(sx)), np.float32(ny) / (np.float32(2) * np.float32(sy)))
    limit = np.float32(np.float64(2.0 / 3.0) * np.float64(half))
    x, y = _k2(nx, sx)[:, None], _k2(ny, sy)[None, :]
    top = float(limit * limit)
    return (x < top) & (y < top) & ((x + y) < top)


def _trans(V, dx, kv, limit, real):
    """exp(i sigma V), band limited."""
    sigma = float(np.float32(1.0) + np.float32(kv) / np.float32(511.0)) * _wavelength(kv)
    t = torch.exp(1j * (V.to(real) * sigma))
    if limit:
        px, py = V.shape[-2:]
        half = min(np.float32(n) / (np.float32(2) * np.float32(np.float32(n) * np.float32(dx))) for n in (px, py))
        top = np.float32(np.float32(2.0) / np.float32(3.0) * half)
        x, y = (_k2(n, np.float32(n) * np.float32(dx)) for n in (px, py))
        t = torch.fft.ifft2(torch.fft.fft2(t) * ((x[:, None] + y[None, :]) < float(top * top)))
    return t


def _propagator(nx, ny, dx, kv, dz, real):
    dx, dz = float(np.float32(dx)), float(np.float32(dz))
    p = []
    for n in (nx, ny):
        i = torch.arange(n, device="cuda", dtype=torch.float64)
        k = torch.where(i > n // 2, i - n, i) / (dx * n)
        p.append(torch.exp(-1j * (math.pi * dz * _wavelength(kv)) * k * k))
    f32 = np.float32
    keep = _band(nx, ny, f32(dx) * f32(nx), f32(dx) * f32(ny))
    P = p[0][:, None] * p[1][None, :] * keep
    return P.to(torch.complex128 if real == torch.float64 else torch.complex64)


def _probe(nx, ny, dx, kv, df0, Cs, real=torch.float64):
    """The probe at the window's centre; df0 and Cs may be tensors with gradients."""
    dx = float(np.float32(dx))
    wl = 12.26 / math.sqrt(kv * 1.0e3 + kv * kv * 0.9788)
    ax, by = nx * dx, ny * dx
    ix, iy = (torch.arange(n, device="cuda", dtype=torch.float64) for n in (nx, ny))
    kx = torch.where(ix > nx // 2, ix - nx, ix)[:, None]
    ky = torch.where(iy > ny // 2, iy - ny, iy)[None, :]
    k2 = kx * kx * (1 / ax) ** 2 + ky * ky * (1 / by) ** 2
    t2 = k2 * wl * wl
    chi = (t2 * df0 / 2 + t2 * t2 * Cs / 4) * (2 * math.pi / wl)
    cx, cy = float(np.float32(nx // 2) * np.float32(dx)), float(np.float32(ny // 2) * np.float32(dx))
    chi = chi - 2 * math.pi * ((ax - cx) * kx / ax + (by - cy) * ky / by)
    inside = k2 <= (math.sin(0.001 * 20.0) / wl) ** 2
    psi = torch.fft.ifft2(torch.where(inside, torch.exp(-1j * chi), torch.zeros_like(chi) + 0j))
    psi = psi * math.sqrt(nx * ny / float((psi.detach().abs() ** 2).sum()))
    return psi.to(torch.complex128 if real == torch.float64 else torch.complex64)


def _through(psi, trans, ipos, config, nx, ny, P, record=None):
    """psi [p][nx][ny] through every slice of trans [config][slice][x][y]."""
    at = [(int(a), int(b)) for a, b in ipos]
    for s in range(trans.shape[1]):
        t = torch.stack([trans[int(config[i]) if config is not None else 0, s, x:x + nx, y:y + ny]
                         for i, (x, y) in enumerate(at)])
        F = torch.fft.fft2(psi * t) * P
        if record is not None:
            record(s, F)
        psi = torch.fft.ifft2(F)
    return psi


def _images(trans, ipos, config, nx, ny, dx, kv, bins, nbins, psi0):
    """Detector images [bin][detector][probe] and total intensities [probe]."""
    wl, f32 = _wavelength(kv), np.float32
    k2 = _k2(nx, f32(dx) * f32(nx))[:, None] + _k2(ny, f32(dx) * f32(ny))[None, :]
    rings = []
    for lo, hi in DETECTORS:
        a, b = (f32(math.sin(f32(v) * 0.001) / wl) for v in (lo, hi))
        rings.append((k2 >= float(a * a)) & (k2 <= float(b * b)))
    P = _propagator(nx, ny, dx, kv, CELL / 2, torch.float64)
    det = np.zeros((nbins, len(DETECTORS), len(ipos)))
    total = np.zeros(len(ipos))
    n2 = float(nx * ny)
    step = max(1, (64 << 20) // (nx * ny * 4))
    for p0 in range(0, len(ipos), step):
        part = slice(p0, min(len(ipos), p0 + step))

        def record(s, F):
            if bins[s] < 0 and s < trans.shape[1] - 1:
                return
            power = F.abs() ** 2 / n2 ** 2
            if bins[s] >= 0:
                for d, ring in enumerate(rings):
                    det[bins[s], d, part] = (power * ring).sum((1, 2)).cpu().numpy()
            total[part] = power.sum((1, 2)).cpu().numpy()

        psi = psi0.expand(part.stop - part.start, nx, ny)
        _through(psi, trans, ipos[part], config[part] if config is not None else None, nx, ny, P, record)
    return det, total


def _power(case, V, ipos, psi0, real):
    """Diffraction intensities [p][n][n] (fractions of the beam) after the last slice."""
    n = case["n"]
    P = _propagator(n, n, case["dx"], case["kv"], CELL / 2, real)
    t = _trans(V, case["dx"], case["kv"], case["limit"], real)[None]
    psi = _through(psi0.expand(len(ipos), n, n), t, ipos, None, n, n, P)
    F = torch.fft.fft2(psi)
    return (F.real ** 2 + F.imag ** 2) / float(n) ** 4


def _start_wave(case, df0, Cs, real):
    if case["kind"] == "probes":
        return _probe(case["n"], case["n"], case["dx"], case["kv"], df0, Cs, real)
    return torch.ones(case["n"], case["n"], device="cuda", dtype=torch.complex128 if real == torch.float64 else torch.complex64)


def _target(case, V, ipos):
    """Measured intensities: the patterns of a specimen that scatters half as much again (an
    early step of a reconstruction)."""
    out = torch.empty(len(ipos), case["n"], case["n"], device="cuda")
    psi0 = _start_wave(case, -50.0, 1.0e4, torch.float32)
    for p in range(0, len(ipos), 256):
        out[p:p + 256] = _power(case, V * 1.5, ipos[p:p + 256], psi0, torch.float32)
    return out


def _gradients(case, seed):
    n, pad = case["n"], case.get("pad", 0)
    V = _potential(seed, case["slices"], n + pad, n + pad, case["dx"])
    ipos = _raster(n, n, pad, case.get("probes", 1))
    target = _target(case, V, ipos)
    V = V.double().requires_grad_()
    df0, Cs = (torch.tensor(v, device="cuda", dtype=torch.float64, requires_grad=True) for v in (-50.0, 1.0e4))
    total = 0.0
    step = max(1, (1 << 22) // (n * n))
    for p in range(0, len(ipos), step):
        I = _power(case, V, ipos[p:p + step], _start_wave(case, df0, Cs, torch.float64), torch.float64)
        loss = ((I - target[p:p + step].double()) ** 2).sum()
        loss.backward()
        total += float(loss.detach())
    out = {"loss": np.float64(total), "V": V.grad}
    return {**out, "df0": df0.grad, "Cs": Cs.grad} if case["kind"] == "probes" else out


def _akima(x, y):
    """Coefficients b, c, d of the Akima spline through (x, y)."""
    m = np.diff(y) / np.diff(x)
    left1 = 2 * m[0] - m[1]
    right1 = 2 * m[-1] - m[-2]
    m = np.concatenate([[2 * left1 - m[0], left1], m, [right1, 2 * right1 - m[-1]]])
    w = np.abs(np.diff(m))
    a, b = w[2:], w[:-2]
    t = np.where(a + b > 1e-25, (a * m[1:-2] + b * m[2:-1]) / np.maximum(a + b, 1e-300), 0.5 * (m[1:-2] + m[2:-1]))
    h, mid = np.diff(x), m[2:-2]
    zero = [0.0]
    return (np.concatenate([t[:-1], zero]), np.concatenate([(3 * mid - 2 * t[:-1] - t[1:]) / h, zero]),
            np.concatenate([(t[:-1] + t[1:] - 2 * mid) / h ** 2, zero]))


def _tapered(table, smax):
    t = table.copy()
    s = t[0]
    s[120:123] = smax, 1.1 * smax, 1.2 * smax
    if s[119] > s[120]:
        for i in range(113):
            if s[119 - i] < s[120] - 0.001 * (i + 1):
                break
            s[119 - i] = s[120] - 0.001 * (i + 1)
            t[1:, 119 - i] = 0
    return t


def _spline(nodes, values, b, c, d, at):
    at = at.contiguous()
    i = torch.searchsorted(nodes, at.reshape(-1), right=True).reshape(at.shape) - 1
    i = torch.where(at <= nodes[0], 0, torch.where(at >= nodes[121], 121, i.clamp(0, 122)))
    z = at - nodes[i]
    return values[i] + (b[i] + (c[i] + d[i] * z) * z) * z


def _profile(nodes, row, qnodes, qrow, geometry):
    """The lookup table [z][r] of one element: f_e summed over q_y, transformed to real
    space, summed over the samples of a slice."""
    nx, nz, sub, dkx, dkz, smax, dz = geometry
    up = lambda v: torch.from_numpy(np.ascontiguousarray(v)).cuda()  # noqa: E731
    coef = tuple(up(v) for v in _akima(nodes, row))
    iz, ix = torch.arange(nz, device="cuda"), torch.arange(nx, device="cuda")
    kz = dkz * torch.where(iz < nz // 2, iz, iz - nz).double()[:, None]
    kx = dkx * torch.where(ix < nx // 2, ix, ix - nx).double()[None, :]
    s2 = kx * kx + kz * kz
    f = _spline(up(nodes), up(row), *coef, s2.sqrt())
    for iy in range(1, nx):
        s3 = (dkx * iy) ** 2 + s2
        keep = s3 < smax * smax
        if not bool(keep.any()):
            break
        f = f + torch.where(keep, 2.0 * _spline(up(qnodes), up(qrow), *coef, s3.sqrt()), 0.0)
    f = torch.where(s2 < smax * smax, f * dkx, 0.0)
    off = (sub - 1) // 2
    real = torch.fft.ifft2(f * torch.exp(1j * kz * (-2.0 * math.pi * (dz / sub * off)))).real * (nx * nz)
    half = torch.zeros(nz // 2 + 2 * off + 1, nx // 2, device="cuda", dtype=torch.float64)
    half[:nz // 2] = real[:nz // 2, :nx // 2]
    sums = sum(half[k:k + nz // 2] for k in range(2 * off + 1))
    return sums.clamp(min=0) * (47.8658 * dkx * dkz / nz)


def _built(case, seed):
    """Projected potential [slices][x][y] of the atoms of an `atoms` case."""
    atoms, offset = _atoms(case, seed)
    f = np.float32
    dx, dz, pot, S = f(case["dx"]), f(CELL / 2), case["n"] + case["pad"], case["slices"]
    R = f(RADIUS)
    rad = int(math.ceil(float(R / dx)))
    nx, radz = 4 * rad, int(math.ceil(float(R / dz)))
    sub = int(math.floor(2 * dz / dx))
    sub += 1 - sub % 2
    nz = 2 * radz * sub
    dkx, dkz = 1.0 / float(f(nx * dx)), sub / float(f(nz * dz))
    smax = 0.5 * nx * dkx / 2.0
    geometry = (nx, nz, sub, dkx, dkz, smax, float(dz))
    tables = [_tapered(np.fromfile("qstem_amd/data/" + n, dtype="<f8").reshape(93, 123), smax)
              for n in ("rez_scatpar_f64.bin", "rez_scatparoffs_f64.bin")]
    V = torch.zeros(S * pot * pot, device="cuda", dtype=torch.float64)
    Nr, Nz, dr = nx // 2, nz // 2, float(f(dx / f(2)))
    box = torch.arange(-rad, rad + 1, device="cuda")
    for Z in sorted(set(atoms[:, 6].astype(int))):
        neutral = _profile(tables[0][0], tables[0][Z], tables[0][0], tables[0][Z], geometry)
        # the ion table's spline, its q_y sum over the neutral table's nodes (the default)
        ion = _profile(tables[1][0], tables[1][Z], tables[0][0], tables[0][Z], geometry)
        mine = atoms[atoms[:, 6] == Z]
        lut = (neutral + float(mine[0, 5]) * ion).reshape(-1)
        px, py = ((mine[:, k].astype(f) - f(offset)) for k in (0, 1))
        pz = (mine[:, 2].astype(f) + f(CELL / 4)).astype(np.float64) - 0.5 * float(dz)
        pz = ((pz.astype(f) - dz) + dz).astype(f)
        iz = np.floor((pz / dz).astype(np.float64) + 0.5).astype(np.int64)
        first = np.maximum(-iz, -radz)
        o = ((iz + first).astype(f) - (pz / dz).astype(f)) * f(sub)
        o = np.trunc(o.astype(np.float64) + 0.5).astype(np.int64)
        for a in range(0, len(mine), 64):
            b = slice(a, a + 64)
            up = lambda v: torch.from_numpy(np.ascontiguousarray(v[b])).cuda()  # noqa: E731
            X, Y = (torch.from_numpy(np.floor((v[b] / dx).astype(np.float64)).astype(np.int64)).cuda()[:, None] + box
                    for v in (px, py))
            inx, iny = (X >= 0) & (X < pot), (Y >= 0) & (Y < pot)
            dX, dY = ((K.float() * float(dx) - up(v)[:, None]).double() for K, v in ((X, px), (Y, py)))
            r = (dX[:, :, None] ** 2 + dY[:, None, :] ** 2).sqrt() / dr
            ir = r.floor().long()
            w = r - ir
            ok = (ir < Nr - 1) & inx[:, :, None] & iny[:, None, :]
            ir = ir.clamp(max=Nr - 2)
            pixel = X.clamp(0, pot - 1)[:, :, None] * pot + Y.clamp(0, pot - 1)[:, None, :]
            z0, zf, zo = up(iz), up(first), up(o)
            for k in range(2 * radz + 1):
                s, z = z0 + zf + k, zo + k * sub
                # the table is even in z, its negative side one row further out
                row = torch.where(z < 0, 1 - z, z)
                good = ok & ((zf + k <= radz) & (s >= 0) & (s < S) & (torch.where(z < 0, -z, z) < Nz - 1))[:, None, None]
                at = row.clamp(0, Nz - 1)[:, None, None] * Nr + ir
                value = torch.where(good, lut[at] * (1 - w) + lut[at + 1] * w, 0.0)
                V.index_add_(0, (s.clamp(0, S - 1)[:, None, None] * pot * pot + pixel).reshape(-1), value.reshape(-1))
    return V.reshape(S, pot, pot)


def exact(case, seed):
    kind, real = case["kind"], torch.float64
    if kind in ("probes", "image"):
        return _gradients(case, seed)
    dx, kv, S = case["dx"], case["kv"], case["slices"]
    if kind == "wave":
        n = case["n"]
        psi = _start_wave(case, 0.0, 0.0, real)[None]
        P = _propagator(n, n, dx, kv, CELL / 2, real)
        V = _potential(seed, S, n, n, dx)
        for s in range(S):
            psi = _through(psi, _trans(V[s:s + 1], dx, kv, case["limit"], real)[None], [(0, 0)], None, n, n, P)
        return {"exit": psi}
    bins, nbins = _bins(S, case.get("every", 0))
    if kind == "atoms":
        n = case["n"]
        V = _built(case, seed)
        t = _trans(V, dx, kv, 0, real)[None]
        ipos = _raster(n, n, case["pad"], case["probes"])
        return {"det": _images(t, ipos, None, n, n, dx, kv, bins, nbins, _probe(n, n, dx, kv, -50.0, 1.0e4))[0]}

    def loaded(px, py, limit):
        return torch.stack([torch.cat([_trans(v[None], dx, kv, limit, real) for v in _potential(seed * 8 + k, S, px, py, dx)])
                            for k in range(case["configs"])])

    if kind == "groups":
        t = loaded(case["pot"], case["pot"], 1)
        return [_images(t, ipos, config, n, n, dx, kv, bins, nbins, _probe(n, n, dx, kv, -50.0, 1.0e4))[0]
                for n, ipos, config in _group_plan(case)]
    nx, ny, pad = case["nx"], case["ny"], case["pad"]
    config = np.arange(case["probes"]) % case["configs"]
    det, total = _images(loaded(nx + pad, ny + pad, case["limit"]), _raster(nx, ny, pad, case["probes"]), config, nx, ny, dx,
                         kv, bins, nbins, _probe(nx, ny, dx, kv, -50.0, 1.0e4))
    return {"det": det, "intensity": total}


def _bins(slices, every):
    """The output bin that each slice leaves as its final value (the last write wins), or -1."""
    every = every if every > 0 else slices
    of = [s // every if s < slices - 1 else slices // every for s in range(slices)]
    last = {b: s for s, b in enumerate(of)}
    return [b if last[b] == s else -1 for s, b in enumerate(of)], slices // every + 1
