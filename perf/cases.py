"""The workloads whose speed is tracked, from the smallest search call to a 256^3 tomogram block.

Each case is one pass through the package's public entry points as a matching program makes it:
exhaustive searches of volumes and images, the Picker class, the squared-difference scorer, the
standalone transforms, and a training pass of the proposal network. listed() gives the fixed cases,
draw() more of the same ranges; exact() restates every path in 64 bits with plain torch.

Left out: ProbabilisticPicker (its score divides by the distance of a noise-driven ratio from 1, so a
change of rounding moves it by any factor), TomoPicker, and the set-up and peak extraction around a
search. Their transforms are the ones timed here.
"""
import math

import numpy as np
import torch

import gtom_amd as gx
from gtom_amd import proposal, tune_micrographs

DEV = "cuda:0"
# Most work of a drawn case: voxel-orientations of a search on a side with fused passes, the same
# divided by the cost of the chirp-z form elsewhere (measured about 20 times), bytes elsewhere.
FUSED_VO = 256 ** 3 * 1152
GENERIC_VO = FUSED_VO // 20


def listed():
    return [
        # One 32^3 sub-tomogram against a coarse set of orientations: the smallest call, all launches.
        dict(name="search_32", kind="search", ndims=3, n=32, box=32, nvol=1, orientations=64, npsi=8, perctf=False),
        # A 64^3 tomogram with the 588 orientations of a 30 degree search (the small configuration of the tests).
        dict(name="search_64", kind="search", ndims=3, n=64, box=32, nvol=1, orientations=588, npsi=12, perctf=False),
        # Eight 96^3 sub-tomograms (3 * 2^a), each with its own defocus: sub-tomogram picking in batches.
        dict(name="search_96x8", kind="search", ndims=3, n=96, box=48, nvol=8, orientations=288, npsi=12, perctf=True),
        # Sub-tomograms of an odd box side, as cropped by hand: no power of two, no Nyquist plane.
        dict(name="search_75x2", kind="search", ndims=3, n=75, box=36, nvol=2, orientations=144, npsi=12, perctf=True),
        # A tomogram binned to 200^3, the side a detector and a binning give.
        dict(name="search_200", kind="search", ndims=3, n=200, box=32, nvol=1, orientations=96, npsi=12, perctf=False),
        # One 256^3 block of a tomogram, 48^3 template, the first 1,152 of 500 x 18 orientations (the benchmark's call).
        dict(name="search_256", kind="search", ndims=3, n=256, box=48, nvol=1, orientations=1152, npsi=18, perctf=False),
        # Sixteen 256^2 particle images against 1,000 central sections (2D branch).
        dict(name="images_256x16", kind="search", ndims=2, n=256, box=64, nvol=16, orientations=1000, npsi=8,
             perctf=False),
        # One 4096^2 micrograph with the autotuned batch (2D branch above 256).
        dict(name="micrograph_4096", kind="search", ndims=2, n=4096, box=64, nvol=1, orientations=192, npsi=8,
             perctf=False),
        # The Picker class: a 128^3 tomogram, a 32^3 reference, 648 orientations.
        dict(name="picker_128", kind="picker", nx=128, ny=128, nz=128, ref=32, orientations=648, npsi=12),
        # Alignment of eight 64^3 sub-tomograms by squared differences over 12^3 shifts.
        dict(name="diff2_64x8", kind="diff2", n=64, box=32, nvol=8, relevant=12, orientations=250),
        # Forward and inverse transforms of a stack of micrographs.
        dict(name="fft_4096x4", kind="fft", ndims=2, nx=4096, ny=4096, nz=1, batch=4),
        # A training pass of the orientation-proposal network (bf16 operands): gradients of 256 tiles.
        dict(name="network_256", kind="network", tiles=256),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _fused(n):
    """Sides up to 256 of the form 2^a or 3 * 2^a."""
    m = n // 3 if n % 3 == 0 else n
    return 8 <= n <= 256 and m & (m - 1) == 0


def draw(rng):
    kind = rng.choice(["search"] * 6 + ["images"] * 2 + ["picker", "diff2", "fft", "network"])
    if kind == "search":
        n = rng.choice([32, 48, 64, 96, 128, 192, 256]) if rng.random() < 0.5 else _log_int(rng, 24, 240)
        box = 2 * rng.randint(6, min(32, n // 2))
        nvol = rng.choice([1, 1, 2, 5]) if n <= 128 else 1
        most = (FUSED_VO if _fused(n) else GENERIC_VO) // (n ** 3 * nvol)
        return dict(kind="search", ndims=3, n=n, box=box, nvol=nvol,
                    orientations=_log_int(rng, 16, max(17, min(1500, most // 2))), npsi=rng.choice([6, 12, 18]),
                    perctf=rng.random() < 0.5)
    if kind == "images":
        n = rng.choice([32, 48, 64, 96, 128, 192, 256, 512, 768, 1024, 2048, 3072, 4096])
        nvol = rng.randint(1, 24) if n <= 256 else rng.randint(1, 3) if n <= 1024 else 1
        most = int(1.2e9) // (n * n * nvol)
        return dict(kind="search", ndims=2, n=n, box=2 * rng.randint(8, min(32, n // 2)), nvol=nvol,
                    orientations=_log_int(rng, 32, max(40, min(2000, most))), npsi=8, perctf=rng.random() < 0.5)
    if kind == "picker":
        nx, ny, nz = (rng.choice([48, 64, 75, 96, 100, 128, 160]) for _ in range(3))
        return dict(kind="picker", nx=nx, ny=ny, nz=nz, ref=rng.choice([16, 24, 30, 32, 48]),
                    orientations=_log_int(rng, 24, 128), npsi=12)
    if kind == "diff2":
        n = rng.choice([24, 32, 48, 64])
        return dict(kind="diff2", n=n, box=2 * rng.randint(6, n // 4), nvol=rng.randint(1, 8),
                    relevant=rng.randint(3, 13), orientations=_log_int(rng, 16, 250))
    if kind == "fft":
        if rng.random() < 0.5:
            return dict(kind="fft", ndims=2, nx=_log_int(rng, 64, 2048), ny=_log_int(rng, 64, 2048), nz=1,
                        batch=rng.randint(1, 6))
        return dict(kind="fft", ndims=3, nx=_log_int(rng, 24, 256), ny=_log_int(rng, 24, 256),
                    nz=_log_int(rng, 24, 256), batch=rng.randint(1, 2))
    return dict(kind="network", tiles=rng.randint(16, 256))


# ---------------------------------------------------------------------------
# inputs, the same for prepare() and exact(): raw float32 data made on the GPU
# ---------------------------------------------------------------------------
def _rotation(a):
    """ZYZ Euler matrices (RELION's layout) of (k, 3) angles, double."""
    a = np.asarray(a, np.float64).reshape(-1, 3)
    (ca, cb, cg), (sa, sb, sg) = np.cos(a).T, np.sin(a).T
    m = np.array([[cg * cb * ca - sg * sa, cg * cb * sa + sg * ca, -cg * sb],
                  [-sg * cb * ca - cg * sa, -sg * cb * sa + cg * ca, sg * sb],
                  [sb * ca, sb * sa, cb]])
    return np.ascontiguousarray(m.transpose(2, 0, 1))


def _angles(count, npsi):
    """Fibonacci-sphere directions times in-plane steps, (rot, tilt, psi) float32."""
    nd = -(-count // npsi)
    i = np.arange(nd)
    a = np.zeros((nd, npsi, 3))
    a[..., 0] = np.mod(i * math.pi * (3 - math.sqrt(5)), 2 * math.pi)[:, None]
    a[..., 1] = np.arccos(1 - (2 * i + 1) / nd)[:, None]
    a[..., 2] = (np.arange(npsi) * 2 * math.pi / npsi)[None]
    return a.reshape(-1, 3)[:count].astype(np.float32)


class _Blobs:
    """A particle: a sum of Gaussians, whose rotated copies are sums of Gaussians again."""

    def __init__(self, box, rng):
        self.box = box
        self.c = rng.uniform(-box / 4, box / 4, (10, 3))
        self.s = rng.uniform(max(0.8, box / 24), max(1.2, box / 12), 10)

    def volume(self, matrix=None, section=False):
        g = torch.arange(self.box, device=DEV, dtype=torch.float32) - self.box // 2
        out = 0
        for c, s in zip(self.c if matrix is None else self.c @ matrix.T, self.s):
            e = [torch.exp(-(g - float(v)) ** 2 / float(2 * s * s)) for v in c]  # x, y, z
            out = out + (e[1][:, None] * e[0] * float(s) if section else e[2][:, None, None] * e[1][:, None] * e[0])
        return out


def _noisy(shape, blobs, rng, gen, copies):
    """Unit Gaussian noise with copies of the particle at random places and orientations."""
    x = torch.randn(shape, device=DEV, generator=gen)
    box = blobs.box
    if min(shape[1:]) < box:
        return x
    for v in range(shape[0]):
        for _ in range(copies):
            m = _rotation(rng.uniform(0, 2 * math.pi, 3))[0]
            at = [int(rng.integers(0, s - box + 1)) for s in shape[1:]]
            x[v][tuple(slice(a, a + box) for a in at)] += 0.5 * blobs.volume(m, section=len(shape) == 3)
    return x


def _raw(case, seed):
    rng = np.random.default_rng(seed)
    gen = torch.Generator(device=DEV)
    gen.manual_seed(seed)
    k = case["kind"]
    if k in ("search", "diff2"):
        n, nv = case["n"], case["nvol"]
        nd = case.get("ndims", 3)
        blobs = _Blobs(case["box"], rng)
        per = k == "diff2" or case["perctf"]
        return dict(template=blobs.volume(), data=_noisy((nv,) + (n,) * nd, blobs, rng, gen, 2 if nd == 3 else 6),
                    defoci=rng.uniform(-4e-6, -2e-6, nv if per else 1),
                    angles=_angles(case["orientations"], case.get("npsi", 10)))
    if k == "picker":
        blobs = _Blobs(case["ref"], rng)
        return dict(ref=blobs.volume(), defoci=rng.uniform(-4e-6, -2e-6, 1),
                    data=_noisy((1, case["nz"], case["ny"], case["nx"]), blobs, rng, gen, 4)[0],
                    angles=_angles(case["orientations"], case["npsi"]))
    if k == "fft":
        shape = (case["batch"],) + (case["nz"],) * (case["ndims"] == 3) + (case["ny"], case["nx"])
        return dict(data=torch.randn(shape, device=DEV, generator=gen))
    n = case["tiles"]
    return dict(tiles=torch.randn((n, 32, 32, 32), device=DEV, generator=gen),
                labels=torch.randint(0, proposal.NCLS, (n,), device=DEV, generator=gen, dtype=torch.int32),
                params=proposal.init_params(seed % 1000))


def _radius(case):
    return max(4.0, case["n"] / 10.0 if case["ndims"] == 3 else case["n"] / 8.0)


OPTICS = dict(pixelsize=10e-10, Cs=2.7e-3, voltage=300e3, amplitude=0.07)


def _ctf(n, nd, defoci):
    if n % 2:  # the library's CTF takes even sides: a program with odd boxes brings its own
        return torch.stack([_ctf64(n, nd, d) for d in defoci]).float()
    return gx.ctf_3d([gx.CtfParams.make(defocus=float(d), **OPTICS) for d in defoci], n, device=DEV, ndims=nd)


def prepare(case, seed):
    r = _raw(case, seed)
    k = case["kind"]
    if k in ("search", "diff2"):
        n, p, nd = case["n"], 2 * case["box"], case.get("ndims", 3)
        s = dict(case=case, projector=gx.prepare_projector(r["template"], p), angles=r["angles"],
                 spectra=gx.d_FFTR2C(r["data"], ndims=nd),
                 ctf=_ctf(n, nd, r["defoci"]))
        if k == "search":
            batch, rows = tune_micrographs.load_table().get(n, (0, gx.ROWS_PLAIN)) if nd == 2 else (0, None)
            s["plan"] = gx.PickPlan(p, n, batch, ndims=nd)
            if nd == 2:
                s["plan"].set_rows_variant(rows)
        return s
    if k == "picker":
        ctf = _ctf(case["ref"], 3, r["defoci"])[0]
        shape = (case["nz"], case["ny"], case["nx"])
        pk = gx.Picker(r["ref"], shape)
        pk.set_image(r["data"], ctf)
        return dict(case=case, picker=pk, angles=r["angles"], best=torch.empty(shape, device=DEV),
                    angle=torch.empty(shape + (3,), device=DEV))
    if k == "fft":
        return dict(case=case, x=r["data"])
    return dict(case=case, net=proposal.ProposalNet(max_tiles=case["tiles"], params=r["params"]), tiles=r["tiles"],
                labels=r["labels"])


def run(s):
    case = s["case"]
    k = case["kind"]
    if k == "search":
        n = case["n"]
        stride = (n // 2 + 1) * n ** (case["ndims"] - 1) if case["perctf"] else 0
        best, index = gx.d_PickSubTomograms(s["plan"], s["projector"], 2.0 * case["box"] / n, s["spectra"], s["ctf"],
                                            s["angles"], _radius(case), ctf_volume_stride=stride)
        return dict(best=best, index=index)
    if k == "picker":
        s["best"].fill_(-1e30)
        s["angle"].zero_()
        s["picker"].perform_correlation(s["best"], s["angle"], angles=s["angles"])
        return dict(best=s["best"], angle=s["angle"])
    if k == "diff2":
        best, index = gx.d_PickSubTomogramsDiff2(s["projector"], 2 * case["box"], 2.0 * case["box"] / case["n"],
                                                 s["spectra"], s["ctf"], (case["relevant"],) * 3, s["angles"])
        return dict(best=best, index=index)
    if k == "fft":
        spectrum = gx.d_FFTR2C(s["x"], ndims=case["ndims"])
        return dict(spectrum=spectrum, back=gx.d_IFFTC2R(spectrum, case["nx"], ndims=case["ndims"]))
    s["net"].load_tiles(s["tiles"])
    gradients, loss = s["net"].gradients(s["labels"])
    return dict(gradients=gradients, loss=loss)


def work(case):
    k = case["kind"]
    if k == "fft":
        points = case["nx"] * case["ny"] * case["nz"] * case["batch"]
        half = points // case["nx"] * (case["nx"] // 2 + 1)
        return dict(bytes=8 * points + 16 * half,
                    flops=5.0 * points * math.log2(case["nx"] * case["ny"] * case["nz"]))
    if k == "network":
        # multiply-adds of the four convolutions and the head, forward and twice that backward
        fwd = 2.0 * 16 * 27 * (32 ** 3 + 16 * 16 ** 3 + 2 * 16 * 8 ** 3) + 2.0 * 1024 * 501
        return dict(bytes=case["tiles"] * (4 * 32 ** 3 + 8) + 8 * proposal.NPARAM, flops=3 * fwd * case["tiles"])
    o = case["orientations"]
    if k == "picker":
        v, vr = case["nx"] * case["ny"] * case["nz"], case["ref"] ** 3
        return dict(bytes=24 * v + 8 * vr, flops=o * (5.0 * v * math.log2(v) + 2.5 * vr * math.log2(vr) + 20.0 * vr))
    nd = case.get("ndims", 3)
    n, nv, p = case["n"], case["nvol"], 2 * case["box"]
    v, h = n ** nd, (n // 2 + 1) * n ** (nd - 1)
    inputs = nv * 8 * h + (nv if k == "diff2" or case["perctf"] else 1) * 4 * h + 4 * p * p * (p + 2)
    if k == "diff2":
        rel = case["relevant"]
        shifts = 8.0 * (rel * h + rel ** 2 * n * (n // 2 + 1) + rel ** 3 * (n // 2 + 1))
        return dict(bytes=inputs + 8 * nv * rel ** 3, flops=nv * o * (shifts + 30.0 * h))
    return dict(bytes=inputs + 8 * nv * v, flops=nv * o * (2.5 * v * math.log2(v) + 20.0 * h))


def tolerance(case):
    k = case["kind"]
    if k == "search":
        return dict(rel=4e-6, max=4e-5, differ=1e-3)
    if k == "picker":
        return dict(rel=1e-2, max=0.9)
    if k == "diff2":
        return dict(rel=1e-5, max=1e-3)
    if k == "fft":
        return dict(rel=4e-6, max=4e-5)
    return dict(rel=2e-2, max=0.5)


# ---------------------------------------------------------------------------
# the same in 64 bits
# ---------------------------------------------------------------------------
def _ctf64(n, nd, defocus):
    k = torch.fft.fftfreq(n, dtype=torch.float64, device=DEV) * n
    k2 = k[:, None] ** 2 + (torch.arange(n // 2 + 1, device=DEV, dtype=torch.float64) ** 2)[None]
    if nd == 3:
        k2 = k[:, None, None] ** 2 + k2[None]
    k2 = k2 / (n * OPTICS["pixelsize"] * 1e10) ** 2
    lam = 12.2643247 / math.sqrt(OPTICS["voltage"] * (1 + OPTICS["voltage"] * 0.978466e-6))
    a = OPTICS["amplitude"]
    # parameters reach the library as 32-bit numbers
    gamma = math.pi * lam * float(np.float32(defocus)) * 1e10 * k2
    gamma = gamma + math.pi / 2 * float(np.float32(OPTICS["Cs"])) * 1e10 * lam ** 3 * k2 ** 2
    return -torch.sin(gamma - math.atan(a / math.sqrt(1 - a * a)))


class _Sections:
    """Trilinear samples of the half spectrum of a padded template at rotated, scaled frequencies."""

    def __init__(self, template, p, n, nd, scale):
        t = template.double()
        b, o = t.shape[0], p // 2 - t.shape[0] // 2
        padded = torch.zeros((p,) * 3, dtype=torch.float64, device=DEV)
        padded[o:o + b, o:o + b, o:o + b] = t
        self.f = torch.fft.fftn(torch.fft.ifftshift(padded)).reshape(-1)
        self.p, self.scale = p, scale
        k = torch.fft.fftfreq(n, dtype=torch.float64, device=DEV) * n
        if n % 2 == 0:
            k[n // 2] = n // 2
        x = torch.arange(n // 2 + 1, device=DEV, dtype=torch.float64)
        g = torch.meshgrid(k, k, x, indexing="ij") if nd == 3 else torch.meshgrid(k, x, indexing="ij")
        z = g[0] if nd == 3 else torch.zeros_like(g[0])
        inside = (g[-1] ** 2 + g[-2] ** 2 + z ** 2 <= (n // 2) ** 2).reshape(-1)
        self.shape, self.at = g[0].shape, inside.nonzero()[:, 0]
        self.k = torch.stack([g[-1].reshape(-1)[self.at], g[-2].reshape(-1)[self.at], z.reshape(-1)[self.at]])

    def __call__(self, angle):
        m = torch.from_numpy(_rotation(angle)[0].T.copy()).to(DEV) * self.scale
        q = m @ self.k
        flip = q[0] < 0
        q = torch.where(flip, -q, q)
        i = torch.floor(q + 1e-9)
        t = q - i
        i = i.long()
        out = 0
        for dz in (0, 1):
            for dy in (0, 1):
                for dx in (0, 1):
                    w = torch.ones_like(t[0])
                    for a, d in ((0, dx), (1, dy), (2, dz)):
                        w = w * (t[a] if d else 1 - t[a])
                    j = (torch.remainder(i[2] + dz, self.p) * self.p + torch.remainder(i[1] + dy, self.p)) * self.p
                    out = out + w * self.f[j + torch.remainder(i[0] + dx, self.p)]
        out = torch.where(flip, out.conj(), out)
        r = torch.zeros(self.shape.numel(), dtype=torch.complex128, device=DEV)
        r[self.at] = out
        return r.reshape(self.shape)


def _local_std64(x, radius):
    dims = x.shape
    d2 = 0
    for a, n in enumerate(dims):
        g = (torch.arange(n, device=DEV, dtype=torch.float64) - n // 2) ** 2
        d2 = d2 + g.reshape((-1,) + (1,) * (len(dims) - 1 - a))
    mask = torch.clamp((torch.cos(torch.clamp(torch.sqrt(d2) - radius, 0, 1) * math.pi) + 1) * 0.5, min=0)
    m = mask.sum()
    f = torch.fft.rfftn(torch.fft.ifftshift(mask)).conj()
    c1 = torch.fft.irfftn(torch.fft.rfftn(x) * f, s=dims)
    c2 = torch.fft.irfftn(torch.fft.rfftn(x * x) * f, s=dims)
    return torch.sqrt(torch.clamp(c2 * m - c1 * c1, min=0)) / m


def _exact_search(case, r):
    n, nd = case["n"], case["ndims"]
    v = n ** nd
    dims = (n,) * nd
    sections = _Sections(r["template"], 2 * case["box"], n, nd, 2.0 * case["box"] / n)
    best, index = [], []
    for j in range(case["nvol"]):
        x = r["data"][j].double()
        e = torch.fft.rfftn(x)
        ctf = _ctf64(n, nd, r["defoci"][j if case["perctf"] else 0])
        top = torch.full(dims, -1e30, dtype=torch.float64, device=DEV)
        at = torch.zeros(dims, dtype=torch.int32, device=DEV)
        for o, a in enumerate(r["angles"]):
            t = torch.fft.irfftn(sections(a) * ctf, s=dims)
            t = torch.fft.rfftn((t - t.mean()) / t.std(correction=0))
            t = t / torch.sqrt((t.real ** 2 + t.imag ** 2).mean())
            c = torch.fft.irfftn(e * t.conj(), s=dims) * v
            better = c > top
            top = torch.where(better, c, top)
            at[better] = o
        best.append(top / _local_std64(x * v, _radius(case)))
        index.append(at)
    return dict(best=torch.stack(best), index=torch.stack(index))


def _exact_picker(case, r):
    nr = case["ref"]
    dims = (case["nz"], case["ny"], case["nx"])
    sections = _Sections(r["ref"], nr, nr, 3, 1.0)
    ctf = _ctf64(nr, 3, r["defoci"][0])
    x = r["data"].double()
    image = torch.fft.rfftn((x - x.mean()) / x.std(correction=0))
    into = []  # where each sample of the reference (origin first) goes in the padded volume
    for n in dims:
        centred = np.arange(n)
        centred = (centred + n // 2) % n + (nr - n - ((nr & (1 - (n & 1))) % 2)) // 2
        keep = (centred >= 0) & (centred < nr)
        into.append((np.nonzero(keep)[0], (centred[keep] + (nr + 1) // 2) % nr))
    to = np.ix_(*[a for a, _ in into])
    of = np.ix_(*[b for _, b in into])
    to, of = ([torch.from_numpy(i).to(DEV) for i in t] for t in (to, of))
    top = torch.full(dims, -1e30, dtype=torch.float64, device=DEV)
    for a in r["angles"]:
        t = torch.zeros(dims, dtype=torch.float64, device=DEV)
        t[tuple(to)] = torch.fft.irfftn(sections(a) * ctf, s=(nr,) * 3)[tuple(of)]
        t = (t - t.mean()) / t.std(correction=0)
        top = torch.maximum(top, torch.fft.irfftn(image * torch.fft.rfftn(t).conj(), s=dims) * top.numel())
    return dict(best=top, angle=None)


def _exact_diff2(case, r):
    n, rel = case["n"], case["relevant"]
    sections = _Sections(r["template"], 2 * case["box"], n, 3, 2.0 * case["box"] / n)
    at = torch.remainder(torch.arange(rel, device=DEV) - rel // 2, n)
    best = []
    for j in range(case["nvol"]):
        e = torch.fft.rfftn(r["data"][j].double())
        ctf = _ctf64(n, 3, r["defoci"][j])
        top = torch.full((rel,) * 3, 1e30, dtype=torch.float64, device=DEV)
        full = torch.zeros((n,) * 3, dtype=torch.complex128, device=DEV)
        for a in r["angles"]:
            t = sections(a) * ctf
            full[..., :n // 2 + 1] = t * e.conj()
            cross = torch.fft.fftn(full).real
            # the shift is -d: exp(-2 pi i k d / n), which fftn's kernel is
            cross = cross[at][:, at][:, :, at]
            top = torch.minimum(top, (t.abs() ** 2).sum() + (e.abs() ** 2).sum() - 2 * cross)
        best.append(top)
    return dict(best=torch.stack(best), index=None)


def _exact_network(case, r):
    p = torch.from_numpy(r["params"]).to(DEV).double().requires_grad_()

    def part(name):
        o, k = proposal.LAYERS[name]
        return p[o:o + k]

    def conv(x, w, b):  # x: (tiles, channels, S, S, S), w: (27, out, in)
        s = x.shape[-1]
        y = torch.nn.functional.pad(x, (1,) * 6)
        out = 0
        for t in range(27):
            z0, y0, x0 = t // 9, t // 3 % 3, t % 3
            v = y[:, :, z0:z0 + s, y0:y0 + s, x0:x0 + s].reshape(x.shape[0], x.shape[1], -1)
            out = out + (v.transpose(1, 2).reshape(-1, x.shape[1]) @ w[t].T)
        out = torch.relu(out + b).reshape(x.shape[0], s ** 3, -1).transpose(1, 2)
        return out.reshape(x.shape[0], -1, s, s, s)

    def pool(x):
        n, c, s = x.shape[:3]
        return x.reshape(n, c, s // 2, 2, s // 2, 2, s // 2, 2).mean((3, 5, 7))

    losses, total = [], 0
    for t, y in zip(r["tiles"].split(32), r["labels"].long().split(32)):
        x = pool(conv(t.double()[:, None], part("w1").reshape(16, 27).T[:, :, None], part("b1")))
        x = pool(conv(x, part("w2").reshape(27, 16, 16), part("b2")))
        x = conv(x, part("w3").reshape(27, 16, 16), part("b3"))
        x = pool(conv(x, part("w4").reshape(27, 16, 16), part("b4")))
        x = x.permute(0, 2, 3, 4, 1).reshape(len(t), -1)
        logits = x @ part("wf").reshape(proposal.NCLS, -1).T + part("bf")
        loss = torch.logsumexp(logits, 1) - logits.gather(1, y[:, None])[:, 0]
        (loss.sum() / case["tiles"]).backward(retain_graph=False)
        losses.append(loss.detach())
    return dict(gradients=p.grad, loss=torch.cat(losses))


def exact(case, seed):
    k = case["kind"]
    if k in ("search", "picker", "diff2"):
        # seconds measured per million voxel-orientations, and about 1 ms a launch-bound orientation
        v = case["n"] ** case.get("ndims", 3) if k != "picker" else case["nx"] * case["ny"] * case["nz"]
        passes = case["orientations"] * case.get("nvol", 1)
        if passes * (2.5e-3 + v * 6e-10) > 20:
            return None
    r = _raw(case, seed)
    if k == "search":
        return _exact_search(case, r)
    if k == "picker":
        return _exact_picker(case, r)
    if k == "diff2":
        return _exact_diff2(case, r)
    if k == "fft":
        dims = tuple(range(-case["ndims"], 0))
        x = r["data"].double()
        return dict(spectrum=torch.fft.rfftn(x, dim=dims), back=x)
    return _exact_network(case, r)
