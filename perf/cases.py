"""Workloads the library's users run, each with its inputs, one pass through the public
modules, the least work a pass needs, and its value in 64-bit arithmetic.

A case is a dict of plain values:
  kind    "fwd" / "adj" (one module call), "pair" (adjoint of forward), "grad" (gradients
          of ||A(x, k) - y||^2 with respect to image and trajectory), "toep" (Toeplitz
          normal operator), "batch" (BatchedKbNufft pair of uneven problems)
  n0, n1, n2   image size (n2 = 0: two-dimensional); the grid is twice that
  batch, coils; sense: coil maps are applied (else the coils are plain channels)
  traj    "radial" (golden angle), "spiral" (variable density), "koosh" (3-D radial);
          shots x reads samples; frames: every batch item has its own trajectory
  j       numpoints, dtype "c64" / "c128", norm "" / "ortho"
  mix     ("batch") which image sizes and shot counts the problems have
"""
import itertools
import math
import random

import numpy as np
import torch

import torchkbnufft_amd as tkbn

L = 2**10  # table oversampling (the modules' default)
KBWIDTH = 2.34


def _case(name, kind, n, batch, coils, traj, shots, reads, sense=False, frames=False, j=6, dtype="c64", norm="", mix=0):
    n = tuple(n) + (0,) * (3 - len(n))
    c = {"kind": kind, "n0": n[0], "n1": n[1], "n2": n[2], "batch": batch, "coils": coils, "traj": traj,
         "shots": shots, "reads": reads, "sense": sense, "frames": frames, "j": j, "dtype": dtype, "norm": norm,
         "mix": mix}
    return dict(c, name=name) if name else c


def listed():
    return [
        # a thumbnail or unit-test sized problem: launches and host work only
        _case("small_64_pair", "pair", (64, 64), 1, 1, "radial", 24, 128),
        # one coil of a single slice, as in the tutorials: 256 x 256, 402 spokes x 512
        _case("single_256_pair", "pair", (256, 256), 1, 1, "radial", 402, 512),
        # the multi-coil slice stack of a SENSE reconstruction, each direction by itself
        _case("sense_320_fwd", "fwd", (320, 320), 4, 16, "radial", 400, 640, sense=True),
        _case("sense_320_adj", "adj", (320, 320), 4, 16, "radial", 400, 640, sense=True),
        # ragged extents, coils and spokes (a grid whose lengths have large prime factors)
        _case("odd_217_pair", "pair", (217, 181), 3, 13, "radial", 171, 433, sense=True, norm="ortho"),
        # dynamic imaging: every frame its own spiral
        _case("frames_192_pair", "pair", (192, 192), 8, 8, "spiral", 16, 1024, sense=True, frames=True),
        # a training step of a trajectory-learning model: image and trajectory gradients
        _case("grad_256", "grad", (256, 256), 1, 12, "spiral", 64, 1536, sense=True),
        # the iterations of a CG-SENSE solver with the Toeplitz operator
        _case("toep_320", "toep", (320, 320), 4, 16, "radial", 400, 640, sense=True),
        # uneven problems served together
        _case("batch_uneven_pair", "batch", (256, 256), 16, 8, "spiral", 48, 1024, mix=3),
        # 3-D radial (kooshball) volumes, each direction by itself
        _case("koosh_160_fwd", "fwd", (160, 160, 160), 1, 8, "koosh", 3200, 512, sense=True),
        _case("koosh_160_adj", "adj", (160, 160, 160), 1, 8, "koosh", 3200, 512, sense=True),
        # double precision, as gradient checks and reference runs use it
        _case("double_128_pair", "pair", (128, 128), 1, 4, "spiral", 16, 1024, dtype="c128"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng: random.Random):
    kind = rng.choice(["pair", "pair", "fwd", "adj", "fwd", "adj", "grad", "toep", "batch", "koosh"])
    j = 6 if rng.random() < 0.8 else 4
    norm = "ortho" if rng.random() < 0.3 else ""
    if kind == "koosh":
        n = _log(rng, 24, 144)
        im = tuple(max(16, n - rng.randrange(0, 1 + n // 6)) for _ in range(3))
        return _case("", rng.choice(["fwd", "adj"]), im, 1, rng.randrange(1, 9), "koosh", _log(rng, 200, 2800),
                     rng.randrange(48, 2 * n + 49), sense=rng.random() < 0.5, j=j, norm=norm)
    n = _log(rng, 48, 320)
    im = (n, n) if rng.random() < 0.5 else (n, max(32, n - rng.randrange(0, 1 + n // 4)))
    reads = rng.randrange(n, 2 * n + 1)
    shots = _log(rng, 8, 400)
    traj = rng.choice(["radial", "spiral"])
    if kind == "batch":
        return _case("", "batch", (256, 256), _log(rng, 4, 20), rng.randrange(1, 13), "spiral", rng.randrange(12, 49),
                     rng.randrange(300, 1100), j=j, mix=rng.randrange(1000))
    if kind == "grad":
        return _case("", "grad", im, 1, rng.randrange(1, 17), traj, min(shots, 250), reads, sense=True, j=j, norm=norm)
    if kind == "toep":
        return _case("", "toep", im, rng.randrange(1, 5), rng.randrange(1, 17), "radial", shots, reads,
                     sense=True, norm=norm)
    sense = rng.random() < 0.7
    batch, coils = rng.randrange(1, 5), _log(rng, 1, 16)
    if rng.random() < 0.15:
        return _case("", kind, im, 1, rng.randrange(1, 7), traj, min(shots, 100), min(reads, 400), sense=sense, j=j,
                     dtype="c128", norm=norm)
    frames = batch > 1 and rng.random() < 0.3
    return _case("", kind, im, batch, coils, traj, shots, reads, sense=sense, frames=frames, j=j, norm=norm)


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _im(case):
    return tuple(case[k] for k in ("n0", "n1", "n2") if case[k])


def _cdtype(case):
    return torch.complex128 if case["dtype"] == "c128" else torch.complex64


def _radial(shots, reads, turn):
    r = -np.pi + 2 * np.pi * np.arange(reads) / reads
    th = np.arange(shots) * np.pi / ((1 + np.sqrt(5)) / 2) + turn
    return np.stack([(np.sin(th)[:, None] * r).reshape(-1), (np.cos(th)[:, None] * r).reshape(-1)])


def _spiral(shots, reads, turn):
    t = np.arange(reads) / reads
    r = np.pi * 0.9999 * t**1.5
    th = 2 * np.pi * 16.0 * t + 2 * np.pi * np.arange(shots)[:, None] / shots + turn
    return np.stack([(r * np.sin(th)).reshape(-1), (r * np.cos(th)).reshape(-1)])


def _koosh(shots, reads, turn):
    i = np.arange(shots) + 0.5
    z = 1 - 2 * i / shots  # spokes uniform on the sphere (golden-angle spiral)
    ph = np.pi * (1 + np.sqrt(5)) * i + turn
    s = np.sqrt(1 - z * z)
    u = np.stack([z, s * np.sin(ph), s * np.cos(ph)])
    r = np.pi * (-1 + 2 * np.arange(reads) / reads)
    return (u[:, :, None] * r).reshape(3, -1)


_TRAJ = {"radial": _radial, "spiral": _spiral, "koosh": _koosh}


def _trajectory(case, seed):
    """(d, M), or (batch, d, M) with a trajectory per frame; rotated by an angle of the seed."""
    turn = np.random.RandomState(seed % (1 << 31)).uniform(0, np.pi)
    f = _TRAJ[case["traj"]]
    if case["frames"]:
        om = np.stack([f(case["shots"], case["reads"], turn + 0.37 * b) for b in range(case["batch"])])
    else:
        om = f(case["shots"], case["reads"], turn)
    return torch.tensor(om, dtype=torch.float64 if case["dtype"] == "c128" else torch.float32)


def _randn(gen, shape, dtype):
    real = torch.float64 if dtype == torch.complex128 else torch.float32
    return torch.view_as_complex(torch.randn(tuple(shape) + (2,), generator=gen, dtype=real, device="cuda"))


def _maps(case, gen):
    """Smooth coil maps of unit root-sum-of-squares: Gaussian profiles with a phase ramp."""
    im = _im(case)
    par = torch.rand((case["batch"], case["coils"], 2 * len(im) + 1), generator=gen, device="cuda", dtype=torch.float64)
    out = None
    for d, n in enumerate(im):
        x = torch.linspace(-1, 1, n, device="cuda", dtype=torch.float64)
        mid = (2.4 * par[..., d] - 1.2)[..., None]
        g = torch.exp(-((x - mid) ** 2) / 1.2) * torch.exp(1j * 2.0 * par[..., len(im) + d][..., None] * x)
        g = g.reshape(g.shape[:2] + (1,) * d + (n,) + (1,) * (len(im) - 1 - d)).to(_cdtype(case))
        out = g if out is None else out * g
    return (out / out.abs().square().sum(1, keepdim=True).sqrt()).contiguous()


def _problems(case, seed):
    """The batch's problems: image size and trajectory of each."""
    r = random.Random(case["mix"])
    out = []
    for p in range(case["batch"]):
        n = r.choice([128, 192, 256])
        one = dict(case, n0=n, n1=n, batch=1, shots=r.randrange(8, case["shots"] + 1))
        out.append((one, _trajectory(one, seed + 7 * p)))
    return out


def _inputs(case, seed):
    """The tensors a program holds before the call, made from the seed alone."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    im, dt = _im(case), _cdtype(case)
    B, C, kind = case["batch"], case["coils"], case["kind"]
    if kind == "batch":
        probs = _problems(case, seed)
        return {"case": case, "problems": probs, "images": [_randn(gen, (1, C) + _im(p), dt) for p, _ in probs]}
    s = {"case": case, "om": _trajectory(case, seed).cuda(), "smaps": _maps(case, gen) if case["sense"] else None,
         "norm": case["norm"] or None}
    if kind == "toep":
        s["kernel"] = _toep_kernel(case, s["om"]).to(dt)
    if kind != "adj":
        s["image"] = _randn(gen, (B, 1 if case["sense"] else C) + im, dt)
    if kind in ("adj", "grad"):
        s["data"] = _randn(gen, (B, C, s["om"].shape[-1]), dt)
    return s


def prepare(case, seed):
    s = _inputs(case, seed)
    im, dt, kind = _im(case), _cdtype(case), case["kind"]
    if kind == "batch":
        s["bt"] = tkbn.BatchedKbNufft([_im(p) for p, _ in s["problems"]], [om for _, om in s["problems"]],
                                      coils=case["coils"], numpoints=case["j"], device=torch.device("cuda"),
                                      autotune=False)
        for buf, x in zip(s["bt"].images, s["images"]):
            buf.copy_(x)
    if kind == "toep":
        s["op"] = tkbn.ToepNufft()
    if kind in ("fwd", "pair", "grad"):
        s["fw"] = tkbn.KbNufft(im_size=im, numpoints=case["j"], dtype=dt).to("cuda")
    if kind in ("adj", "pair"):
        s["ad"] = tkbn.KbNufftAdjoint(im_size=im, numpoints=case["j"], dtype=dt).to("cuda")
    return s


def run(s):
    kind = s["case"]["kind"]
    if kind == "batch":
        images = s["bt"].pair()
        return {"images": list(images), "kdata": list(s["bt"].kdata)}
    if kind == "toep":
        return s["op"](s["image"], s["kernel"], smaps=s["smaps"], norm=s["norm"])
    if kind == "fwd":
        return s["fw"](s["image"], s["om"], smaps=s["smaps"], norm=s["norm"])
    if kind == "adj":
        return s["ad"](s["data"], s["om"], smaps=s["smaps"], norm=s["norm"])
    if kind == "pair":
        kdata = s["fw"](s["image"], s["om"], smaps=s["smaps"], norm=s["norm"])
        return {"kdata": kdata, "image": s["ad"](kdata, s["om"], smaps=s["smaps"], norm=s["norm"])}
    x = s["image"].clone().requires_grad_(True)
    k = s["om"].clone().requires_grad_(True)
    loss = torch.sum(torch.abs(s["fw"](x, k, smaps=s["smaps"], norm=s["norm"]) - s["data"]) ** 2)
    loss.backward()
    return {"loss": loss.detach(), "image": x.grad, "ktraj": k.grad}


# ---------------------------------------------------------------------------
# the least work of a pass: inputs read once, outputs written once; the FFTs and taps
# ---------------------------------------------------------------------------
def work(case):
    if case["kind"] == "batch":
        ws = [work(dict(p, kind="pair", sense=False)) for p, _ in _problems(case, 0)]
        return {k: sum(w[k] for w in ws) for k in ("bytes", "flops")}
    im = _im(case)
    d, B, C = len(im), case["batch"], case["coils"]
    el = 16 if case["dtype"] == "c128" else 8
    P, G, M = math.prod(im), math.prod(2 * n for n in im), case["shots"] * case["reads"]
    image = B * (1 if case["sense"] else C) * P * el
    maps = B * C * P * el if case["sense"] else 0
    traj = (B if case["frames"] else 1) * d * M * el // 2
    data = B * C * M * el
    fft = 5 * B * C * G * math.log2(G)
    taps = 4 * B * C * M * case["j"] ** d
    passes = {"fwd": 1, "adj": 1, "pair": 2, "grad": 2, "toep": 2}[case["kind"]]
    if case["kind"] == "toep":
        return {"bytes": 2 * image + maps + G * el, "flops": 2 * fft}
    extra = image + traj if case["kind"] in ("grad", "pair") else 0
    if case["kind"] == "grad":
        taps *= 2  # the trajectory's gradient takes the taps once more
    return {"bytes": image + maps + traj + data + extra, "flops": passes * (fft + taps)}


# ---------------------------------------------------------------------------
# the same quantities in 64 bits, in plain torch.  The table path reads table entry
# round((tm - k) L) of sample tm = omega / gam in the precision of the trajectory; the
# entries, phases and all sums are 64-bit here.
# ---------------------------------------------------------------------------
def _table64(n, k, j):
    u = torch.arange(j * L + 1, dtype=torch.float64) / L - j / 2
    alpha = torch.tensor(KBWIDTH * j, dtype=torch.float64)
    a = alpha * torch.sqrt((1 - (u / (j / 2)) ** 2).clamp(min=0))
    kb = torch.special.i0(a) / torch.special.i0(alpha)
    kb[0] = kb[-1] = 0
    return torch.polar(kb, -math.pi * (n - 1) / k * u)


def _apod64(im, j):
    alpha = KBWIDTH * j
    i0 = torch.special.i0(torch.tensor(alpha, dtype=torch.float64))
    out = torch.ones((), dtype=torch.float64)
    for d, n in enumerate(im):
        w = (torch.arange(n, dtype=torch.float64) - (n - 1) / 2) / (2 * n)
        y = torch.sqrt(alpha**2 - (math.pi * j * w) ** 2)
        out = out[..., None] * (i0 / j * y / torch.sinh(y))
    return out.cuda()


def _taps64(im, shift, om, j, derivative=False):
    """Per dimension: grid indices (j, M), weights (j, M) and, asked for, their derivatives
    with respect to the tap distance; and the phase (M) of the samples om (d, M)."""
    om = om.detach().cpu()
    real = om.dtype
    out, theta = [], torch.zeros(om.shape[-1], dtype=real)
    for d, n in enumerate(im):
        k = 2 * n
        gam = (torch.tensor(1, dtype=real) / k) * torch.tensor(2 * math.pi, dtype=real)
        tm = om[d] / gam.expand_as(om[d])
        base = torch.floor(tm - j / 2).to(torch.int64) + 1
        idx = base[None] + torch.arange(j)[:, None]
        ul = (tm[None] - idx.to(real)) * L
        r = torch.round(ul)
        ti = (r.to(torch.int64) + (j * L) // 2).clamp(0, j * L)
        tab = _table64(n, k, j)
        w = tab[ti].cuda()
        dw = None
        if derivative:  # of the quadratic through the three entries around the tap
            ext = torch.cat([tab.new_zeros(1), tab, tab.new_zeros(1)])
            lo, hi = ext[ti], ext[ti + 2]
            fr = (ul - r).double()
            dw = (((hi - lo) * 0.5 + fr * (hi - 2 * tab[ti] + lo)) * L / float(gam)).cuda()
        theta = theta + om[d] * torch.tensor(shift[d], dtype=real)
        out.append((torch.remainder(idx, k).cuda(), w, dw))
    theta = theta.double().cuda()
    return out, torch.polar(torch.ones_like(theta), theta)


def _each_tap(taps, im):
    """Flattened grid index and the taps of every dimension, tap by tap."""
    for js in itertools.product(*[range(t[0].shape[0]) for t in taps]):
        flat = 0
        for d, q in enumerate(js):
            flat = flat * (2 * im[d]) + taps[d][0][q]
        yield flat, js


def _interp64(grid, taps, phase, im):
    """(rows, *K) -> (rows, M)"""
    g = grid.reshape(grid.shape[0], -1)
    out = torch.zeros((g.shape[0], phase.shape[0]), dtype=torch.complex128, device="cuda")
    for flat, js in _each_tap(taps, im):
        w = phase
        for d, q in enumerate(js):
            w = w * taps[d][1][q]
        out += w * g[:, flat]
    return out


def _spread64(data, taps, phase, im):
    """(rows, M) -> (rows, *K)"""
    rows = data.shape[0]
    grid = torch.zeros((rows, math.prod(2 * n for n in im), 2), dtype=torch.float64, device="cuda")
    for flat, js in _each_tap(taps, im):
        w = phase
        for d, q in enumerate(js):
            w = w * taps[d][1][q]
        grid.index_add_(1, flat, torch.view_as_real(data * w.conj()))
    return torch.view_as_complex(grid).reshape((rows,) + tuple(2 * n for n in im))


def _scale64(im, norm):
    return 1 / math.sqrt(math.prod(2 * n for n in im)) if norm == "ortho" else 1.0


def _to_grid64(x, im, j, norm):
    x = x * _apod64(im, j)
    return torch.fft.fftn(x, s=[2 * n for n in im], dim=list(range(-len(im), 0))) * _scale64(im, norm)


def _from_grid64(grid, im, j, norm):
    x = torch.fft.ifftn(grid, dim=list(range(-len(im), 0)), norm="forward")
    x = x[(Ellipsis,) + tuple(slice(0, n) for n in im)]
    return x * _apod64(im, j) * _scale64(im, norm)


def _toep_kernel(case, om):
    """Kernel of the normal operator on the doubled grid: the FFT of the trajectory's
    point-spread function (an adjoint NUFFT of ones onto lags -n .. n - 1)."""
    im = _im(case)
    big = tuple(2 * n for n in im)
    taps, phase = _taps64(big, im, om, case["j"])
    psf = _from_grid64(_spread64(torch.ones_like(phase)[None], taps, phase, big), big, case["j"], "")[0]
    dims = list(range(len(im)))
    kernel = torch.fft.fftn(torch.fft.ifftshift(psf, dim=dims), dim=dims) / math.prod(big)
    return kernel.real.to(torch.complex128)


def _rows64(case, s, b):
    """Coil images (C, *im) of batch item b in 64 bits."""
    x = s["image"][b].to(torch.complex128)
    return x * s["smaps"][b].to(torch.complex128) if case["sense"] else x


def _combine64(case, s, b, x):
    return (x * s["smaps"][b].to(torch.complex128).conj()).sum(0, keepdim=True) if case["sense"] else x


def exact(case, seed):
    im, j = _im(case), case["j"]
    shift = [n // 2 for n in im]
    s = _inputs(case, seed)
    if case["kind"] == "batch":
        images, kdata = [], []
        for (one, om), x in zip(s["problems"], s["images"]):
            n = _im(one)
            taps, phase = _taps64(n, [v // 2 for v in n], om, j)
            y = _interp64(_to_grid64(x[0].to(torch.complex128), n, j, ""), taps, phase, n)
            kdata.append(y[None])
            images.append(_from_grid64(_spread64(y, taps, phase, n), n, j, "")[None])
        return {"images": images, "kdata": kdata}
    norm = case["norm"]
    if case["kind"] == "toep":
        # norm "ortho" scales each transform by 1 / sqrt(prod K), none leaves both unscaled
        scale = _scale64(im, norm) ** 2
        kernel = s["kernel"].to(torch.complex128)
        dims, out = list(range(-len(im), 0)), []
        for b in range(case["batch"]):
            f = torch.fft.fftn(_rows64(case, s, b), s=[2 * n for n in im], dim=dims) * kernel
            x = torch.fft.ifftn(f, dim=dims, norm="forward")[(Ellipsis,) + tuple(slice(0, n) for n in im)] * scale
            out.append(_combine64(case, s, b, x))
        return torch.stack(out)
    kdata, images = [], []
    taps = None
    for b in range(case["batch"]):
        if taps is None or case["frames"]:
            om = s["om"][b] if case["frames"] else s["om"]
            taps, phase = _taps64(im, shift, om, j, derivative=case["kind"] == "grad")
        y = None
        if case["kind"] != "adj":
            grid = _to_grid64(_rows64(case, s, b), im, j, norm)
            y = _interp64(grid, taps, phase, im)
            kdata.append(y)
        if case["kind"] in ("adj", "pair"):
            y = y if y is not None else s["data"][b].to(torch.complex128)
            images.append(_combine64(case, s, b, _from_grid64(_spread64(y, taps, phase, im), im, j, norm)))
    if case["kind"] == "fwd":
        return torch.stack(kdata)
    if case["kind"] == "adj":
        return torch.stack(images)
    if case["kind"] == "pair":
        return {"kdata": torch.stack(kdata), "image": torch.stack(images)}
    # gradients of sum |y - data|^2 (one batch item)
    r = kdata[0] - s["data"][0].to(torch.complex128)
    gi = _combine64(case, s, 0, _from_grid64(_spread64(2 * r, taps, phase, im), im, j, norm))
    flat = grid.reshape(grid.shape[0], -1)
    q = (2 * r).conj() * phase
    gk = []
    for d in range(len(im)):
        mixed = [(t[0], t[2] if e == d else t[1], None) for e, t in enumerate(taps)]
        sums = _interp64(flat, mixed, torch.ones_like(phase), im)
        gk.append((q * sums).real.sum(0) - shift[d] * (q * _interp64(flat, taps, torch.ones_like(phase), im)).imag.sum(0))
    return {"loss": r.abs().square().sum(), "image": gi[None], "ktraj": torch.stack(gk)}
