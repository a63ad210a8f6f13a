"""The calls whose time counts: invert, predict, planning and weighting at the
sizes users image at, as plain dicts, with the inputs, one pass, the
unavoidable work, the tolerance and a 64-bit evaluation of each.

A case names an `op`, the way a program uses the framework:

  cycle    image weights (unless "none"), plan, invert, predict on new samples
  invert   plan and invert (a dirty image or PSF of new samples)
  predict  predict with a kept plan
  major    invert and predict with a kept plan (a later major cycle)
  facets   invert and predict of a facet set, one captured graph per direction
  grad     chi^2 of the differentiable degridding and its gradient
  host     the host-array protocol of WStackingGridder, one pass, both ways
  direct   the FP64 direct transform, both ways

Observations are arrays of `antennas` stations over `times` integrations and
`channels` channels (wsclean_amd.synth); `extent` is the longest baseline times
the pixel size (0.5: the edge of the uv grid). Four images are XX, XY, YX, YY
with XY and YX complex; one or two are real.
"""
import math

import numpy as np
import torch

import wsclean_amd
from wsclean_amd import synth
from wsclean_amd.autograd import WStackingOperator, chi_squared, degrid
from wsclean_amd.direct import direct_invert, direct_predict
from wsclean_amd.facets import FacetBatch
from wsclean_amd.weights import DeviceImageWeights

KERNEL = 7
DEFAULTS = dict(op="cycle", width=1024, height=1024, layers=32, antennas=64, times=100,
                channels=16, dt=10.0, radius=3000.0, spiral=False, extent=0.45, images=1,
                precision="mixed", oversampling=63, weighting="none", facets=0,
                field=404)


def _case(**kw):
    c = dict(DEFAULTS)
    c.update(kw)
    return c


def listed():
    return [
        # a snapshot's quick look: one integration, where launches and host
        # synchronisation count
        _case(name="snapshot-256", width=256, height=256, layers=8, times=1,
              weighting="natural"),
        # the ordinary dirty image: 2016 baselines, 3.2M samples, Stokes I
        _case(name="dirty-1024", op="invert"),
        # the model visibilities of the same observation, plan kept
        _case(name="predict-1024", op="predict"),
        # the reference's class driven from host arrays at its default
        # precision and oversampling
        _case(name="host-1024", op="host", times=20, precision="reference", oversampling=1023),
        # a gradient step on a model image through the degridding
        _case(name="grad-512", op="grad", width=512, height=512, layers=16, times=40),
        # a later major cycle of four correlations at 2048^2
        _case(name="major-2048", op="major", width=2048, height=2048, images=4, antennas=62,
              times=225, channels=32, dt=16.0, radius=20000.0, spiral=True),
        # an odd field: neither square nor a power of two, two polarisations,
        # uniform weighting
        _case(name="odd-1500x1260", width=1500, height=1260, layers=24, images=2, antennas=48,
              times=120, channels=24, weighting="uniform"),
        # the reference's arithmetic on the device, two polarisations
        _case(name="reference-2048", op="major", width=2048, height=2048, images=2,
              precision="reference", antennas=62, times=120, channels=32, dt=16.0,
              radius=20000.0, spiral=True),
        # 16 uneven facets of one major cycle
        _case(name="facets-16", op="facets", facets=16, width=2048, height=2048, images=4,
              antennas=62, times=112, channels=64, dt=32.0, radius=40000.0, spiral=True,
              layers=0),
        # Stokes I gridded at a padded size and large oversampling, the
        # setting for accurate wide images
        _case(name="padded-6144", width=6144, height=6144, layers=96, oversampling=1023,
              antennas=62, times=450, channels=64, dt=8.0, radius=40000.0, spiral=True,
              extent=0.6, weighting="briggs"),
        # a long observation in four correlations: the whole step
        _case(name="cycle-4096", width=4096, height=4096, layers=64, images=4, antennas=62,
              times=1800, channels=64, dt=2.0, radius=40000.0, spiral=True, extent=0.85,
              weighting="briggs"),
        # the FP64 direct transform of a small field
        _case(name="direct-512", op="direct", width=512, height=512, layers=0, antennas=32,
              times=4, channels=8),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _smooth(n, multiple):
    """The smallest multiple of `multiple` from n up with no prime above 7."""
    n = -(-n // multiple) * multiple
    while True:
        m = n
        for p in (2, 3, 5, 7):
            while m % p == 0:
                m //= p
        if m == 1:
            return n
        n += multiple


def _size(rng, lo, hi):
    """A size that a uv tile divides, spread over the logarithm."""
    return _smooth(_log_int(rng, lo, hi), rng.choice((8, 16, 16, 32, 64, 60)))


def draw(rng):
    op = rng.choice(("cycle", "cycle", "invert", "predict", "major", "major", "facets", "grad",
                     "host", "direct"))
    images = rng.choice((1, 1, 2, 4))
    if op == "direct":
        n = _log_int(rng, 64, 256) * 2
        return _case(op=op, width=n, height=n, layers=0, antennas=rng.randint(8, 32),
                     times=rng.randint(1, 4), channels=rng.randint(1, 8))
    if op == "facets":
        n = _size(rng, 256, 1024)
        return _case(op=op, facets=rng.randint(3, 10), field=rng.randint(1, 10 ** 6),
                     width=n, height=n, images=images,
                     antennas=rng.randint(24, 62), times=_log_int(rng, 10, 60),
                     channels=rng.randint(4, 32), dt=32.0, radius=20000.0, spiral=True, layers=0)
    width = _size(rng, 128, 3072)
    height = width
    if rng.random() < 0.3:
        # the same tile divides both sides
        multiple = 60 if width % 60 == 0 else math.gcd(width, 64)
        height = _smooth(_log_int(rng, 128, width), multiple)
    c = _case(op=op, width=width, height=height, layers=_log_int(rng, 4, 96),
              antennas=rng.randint(16, 64), times=_log_int(rng, 1, 200),
              channels=_log_int(rng, 1, 64), images=images,
              precision=rng.choice(("mixed", "mixed", "mixed", "reference")),
              oversampling=rng.choice((63, 63, 63, 1023)),
              extent=rng.choice((0.45, 0.45, 0.6)),
              spiral=rng.random() < 0.5)
    if c["spiral"]:
        c["radius"] = float(_log_int(rng, 5000, 40000))
    if op == "cycle":
        c["weighting"] = rng.choice(("none", "natural", "uniform", "briggs"))
    if op in ("grad", "host"):
        c["images"] = 1
    if op == "host":
        c["times"] = min(c["times"], 20)
    return c


# ------------------------------------------------------------------ inputs
def _observation(case, seed):
    rng = np.random.default_rng([seed, 1])
    make = synth.log_spiral_array if case["spiral"] else synth.disc_array
    enu = make(case["antennas"], case["radius"], rng)
    freqs = np.linspace(120e6, 168e6, case["channels"])
    return synth.observe(enu, -26.70, -30.0, case["times"], case["dt"], freqs)


def _geometry(case, obs):
    """Pixel size and w limits (wavelengths) of the observation."""
    wl = obs.wavelengths
    longest = float(np.sqrt((obs.uvw_m ** 2).sum(axis=1)).max())
    pixel = case["extent"] * float(wl.min()) / longest
    aw = np.abs(obs.uvw_m[:, 2])
    return pixel, float(aw.min() / wl.max()), float(aw.max() / wl.min())


def _complex(case):
    return (1, 2) if case["images"] == 4 else ()


def _gen(seed, dev):
    g = torch.Generator(device=dev)
    g.manual_seed(int(seed))
    return g


def _model(n_images, height, width, gen, dev):
    """A clean model: point components of log-uniform flux."""
    m = torch.zeros((n_images, height * width), dtype=torch.float32, device=dev)
    n = max(16, width * height // 4096)
    for i in range(n_images):
        at = torch.randint(0, height * width, (n,), generator=gen, device=dev)
        flux = torch.exp(torch.rand((n,), generator=gen, device=dev) * 6.9 - 4.6)
        m[i].scatter_reduce_(0, at, flux, "amax")  # (components may coincide)
    return m.reshape(n_images, height, width)


def _visibilities(nrow, nchan, images, gen, dev):
    """Noise about a source at the phase centre."""
    v = torch.randn((nrow, nchan, images), dtype=torch.complex64, device=dev, generator=gen)
    v += 1.0
    return v


def _facet_set(case):
    # boxes between a quarter of the size and the size, within 2.5 degrees
    return synth.config4_facets(seed=case["field"], n=case["facets"], lo=case["width"] // 4,
                                hi=case["width"], radius_deg=2.5)


FACET_PIXEL = 4.0 * synth.ARCSEC


def _inputs(case, seed):
    """Everything that is made from the seed, on the device."""
    dev = torch.device("cuda", 0)
    obs = _observation(case, seed)
    pixel, min_w, max_w = _geometry(case, obs)
    gen = _gen(seed, dev)
    s = dict(case=case, dev=dev, obs=obs, pixel=pixel, min_w=min_w, max_w=max_w,
             uvw=torch.from_numpy(obs.uvw_m).to(dev),
             wl=torch.from_numpy(np.ascontiguousarray(obs.wavelengths)).to(dev))
    nrow, nchan, n = obs.nrow, obs.nchan, case["images"]
    op = case["op"]
    if op != "predict":
        s["vis"] = _visibilities(nrow, nchan, n, gen, dev)
    if case["weighting"] != "none":
        s["weights"] = torch.rand((nrow, nchan, n), dtype=torch.float32, device=dev,
                                  generator=gen) + 0.5
    if op == "facets":
        s["facets"] = _facet_set(case)
        s["model"] = [_model(n, f.height, f.width, gen, dev) for f in s["facets"]]
        s["model_im"] = [m.roll(1, 2) for m in s["model"]] if _complex(case) else None
    elif op != "invert":
        s["model"] = _model(n, case["height"], case["width"], gen, dev)
        s["model_im"] = s["model"].roll(1, 2) if _complex(case) else None
    return s


def prepare(case, seed):
    s = _inputs(case, seed)
    dev, op, n = s["dev"], case["op"], case["images"]
    w, h = case["width"], case["height"]
    nrow, nchan = s["obs"].nrow, s["obs"].nchan
    if op == "direct":
        return s
    if op == "host":
        s["uvw_host"], s["wl_host"] = s["obs"].uvw_m, s["obs"].wavelengths
        s["vis_host"] = s["vis"].cpu().numpy()
        s["model_host"] = s["model"].cpu().numpy()
        s["g"] = wsclean_amd.WStackingGridder(w, h, s["pixel"], s["pixel"], KERNEL,
                                              case["oversampling"], precision=case["precision"])
        s["g"].prepare_w_layers(case["layers"], 0.0, s["min_w"], s["max_w"])
        return s
    if op == "grad":
        s["op"] = WStackingOperator(w, h, s["pixel"], s["pixel"], s["uvw"], s["wl"],
                                    case["layers"], kernel_size=KERNEL,
                                    oversampling=case["oversampling"],
                                    precision=case["precision"])
        return s
    if op == "facets":
        fb = FacetBatch(s["facets"], FACET_PIXEL, FACET_PIXEL, s["uvw"], s["wl"], n_images=n,
                        complex_images=_complex(case), kernel_size=KERNEL,
                        precision=case["precision"], oversampling=case["oversampling"])
        s["fb"], s["re"] = fb, fb.images()
        s["im"] = fb.images() if _complex(case) else None
        s["out"] = [torch.empty((nrow, nchan, n), dtype=torch.complex64, device=dev)
                    for _ in s["facets"]]
        s["invert"] = fb.capture_invert(s["vis"], 1.0 / (nrow * nchan), s["re"], s["im"])
        s["predict"] = fb.capture_predict(s["model"], s["model_im"], s["out"])
        return s
    g = wsclean_amd.DeviceGridder(w, h, s["pixel"], s["pixel"], KERNEL, case["oversampling"],
                                  precision=case["precision"], n_images=n,
                                  complex_images=_complex(case))
    g.prepare_w_layers(case["layers"], s["min_w"], s["max_w"])
    s["g"] = g
    if op != "predict":
        s["re"] = torch.zeros((n, h, w), dtype=torch.float32, device=dev)
        s["im"] = torch.zeros_like(s["re"]) if _complex(case) else None
    if op != "invert":
        s["out"] = torch.empty((nrow, nchan, n), dtype=torch.complex64, device=dev)
    if case["weighting"] != "none":
        s["weights_xx"] = s["weights"][..., :1].contiguous()
    if op in ("predict", "major"):
        g.plan(s["uvw"], s["wl"])
    return s


def _factor(s):
    """1 / (sum of weights) for unit weights; weighted images are normalised
    by their own weight sums."""
    return 1.0 if s["case"]["weighting"] != "none" else 1.0 / (s["obs"].nrow * s["obs"].nchan)


def run(s):
    case, op = s["case"], s["case"]["op"]
    if op == "direct":
        img = direct_invert(s["uvw"], s["wl"], s["vis"], case["width"], case["height"],
                            s["pixel"], s["pixel"], multiplication_factor=_factor(s))
        out = direct_predict(s["model"][0], s["uvw"], s["wl"], s["pixel"], s["pixel"])
        return {"image": img, "vis": out}
    if op == "host":
        g = s["g"]
        for p in range(g.n_passes):
            g.start_inversion_pass(p)
            g.add_data(s["uvw_host"], s["wl_host"], s["vis_host"])
            g.finish_inversion_pass()
        re, _ = g.finalize_image(_factor(s))
        g.initialize_prediction(s["model_host"])
        for p in range(g.n_passes):
            g.start_prediction_pass(p)
            out = g.sample_data(s["uvw_host"], s["wl_host"])
        return {"image": re, "vis": out}
    if op == "grad":
        x = s["model"][0].clone().requires_grad_(True)
        vis = degrid(x, s["op"])
        loss = chi_squared(vis, s["vis"][..., 0])
        loss.backward()
        return {"vis": vis.detach(), "loss": loss.detach(), "grad": x.grad}
    if op == "facets":
        s["invert"].launch()
        s["predict"].launch()
        return {"re": s["re"], "im": s["im"], "vis": s["out"]}
    g = s["g"]
    if case["weighting"] != "none":
        iw = DeviceImageWeights(case["weighting"], case["width"], case["height"], s["pixel"],
                                s["pixel"], robust=0.0)
        iw.grid(s["uvw"], s["wl"], s["weights_xx"])
        iw.finish()
        g.set_weighting(iw, s["weights"], "normal")
        s["image_weights"] = iw  # the previous pass's are released after the new ones are set
    got = {}
    if op in ("cycle", "invert"):
        g.plan(s["uvw"], s["wl"])
    if op != "predict":
        g.invert(s["vis"], _factor(s), s["re"], s["im"])
        got["re"], got["im"] = s["re"], s["im"]
    if op != "invert":
        g.predict(s["model"], s["model_im"], s["out"])
        got["vis"] = s["out"]
    return got


# ------------------------------------------------- unavoidable work, tolerance
def _samples(case):
    return case["antennas"] * (case["antennas"] - 1) // 2 * case["times"], case["channels"]


def work(case):
    """Inputs read and outputs written once; K x K taps of a complex value by a
    real kernel per visibility, 5 N log2 N per layer transform, 8 per layer
    cell for the w terms."""
    rows, nchan = _samples(case)
    vis, n, op = rows * nchan * case["images"], case["images"], case["op"]
    pixels = case["width"] * case["height"]
    if op == "direct":
        return {"bytes": rows * 24 + vis * 16 + pixels * 12,
                "flops": 16.0 * rows * nchan * (pixels + max(16, pixels // 4096))}
    planes = n + len(_complex(case))
    ways = 1 if op in ("invert", "predict") else 2
    flops = ways * vis * 4.0 * KERNEL * KERNEL
    nbytes = rows * 24 + ways * (8 * vis + 4 * planes * pixels)
    if case["weighting"] != "none":
        nbytes += 4 * vis
    if op == "facets":
        # facet sides average 5/8 of the largest, layers about 30
        mean = 25.0 / 64.0 * pixels
        flops = case["facets"] * (flops + ways * 30 * n * mean * (5 * math.log2(mean) + 8))
        nbytes = rows * 24 + 8 * vis * (1 + case["facets"]) + \
            case["facets"] * ways * 4 * planes * mean
    else:
        flops += ways * case["layers"] * n * pixels * (5 * math.log2(pixels) + 8)
    return {"bytes": float(nbytes), "flops": float(flops)}


def tolerance(case):
    """32-bit tables, products, transforms and sums: about four times what
    separates the path from the 64-bit evaluation below (3e-7), the largest
    single difference lying in the tail of millions of values (2e-5 between
    two plans of the same samples, whose sums run in another order). The FP64
    direct transform differs by the rounding of its visibilities to 32 bits."""
    if case["op"] == "direct":
        return {"rel": 1e-7, "max": 5e-7}
    return {"rel": 1.2e-6, "max": 1e-4}


# --------------------------------------------------------- 64-bit evaluation
def _kernel_1d(os):
    """The Kaiser-Bessel times sinc table, k1d[x * os + i] at tap x and
    fractional offset i."""
    n = os * KERNEL
    mid = n // 2
    i = np.arange(mid + 1, dtype=np.float64)
    x = np.where(i == 0, 1.0, i)
    sinc = np.where(i == 0, 1.0 / os, np.sin(np.pi * x / os) / (np.pi * x))
    half = sinc * np.i0(8.6 * np.sqrt(1.0 - (i / mid) ** 2)) * os / np.i0(8.6)
    k = np.zeros(n)
    k[mid:2 * mid + 1] = half[:n - mid]
    k[:mid] = k[n - 1 - np.arange(mid)]
    return k


def _correction(k1d, os, axis, dev):
    """The kernel's transform at pixel offsets 0..axis/2, half a sample off
    (a REDFT01)."""
    n = axis * os // 2
    half = KERNEL * os // 2
    h = torch.from_numpy(k1d[half + np.arange(half + 1)[:min(half + 1, n)]]).to(dev)
    k = torch.arange(axis // 2 + 1, dtype=torch.float64, device=dev) + 0.5
    acc = torch.full_like(k, float(h[0]))
    for j0 in range(1, h.numel(), 512):
        j = torch.arange(j0, min(j0 + 512, h.numel()), dtype=torch.float64, device=dev)
        acc += 2.0 * (torch.cos(math.pi / n * k[:, None] * j[None, :]) @ h[j0:j0 + j.numel()])
    x = torch.arange(axis, device=dev)
    return acc[(x - axis // 2).abs()]


class _Exact:
    """The w-stacking map of one image kind in 64 bits."""

    def __init__(self, w, h, pixel, layers, min_w, max_w, os, cplx, uvw, wl, l0=0.0, m0=0.0,
                 rotate=False):
        self.w, self.h, self.nw, self.cplx = w, h, layers, cplx
        self.dev = dev = uvw.device
        if min_w == max_w:
            max_w += 1.0
        k1d = _kernel_1d(os)
        # table row p holds k1d[x * os + os - 1 - p]
        tab = np.ascontiguousarray(k1d.reshape(KERNEL, os)[:, ::-1].T)
        self.tab = torch.from_numpy(tab).to(dev)
        self.corr = _correction(k1d, os, h, dev)[:, None] * _correction(k1d, os, w, dev)[None, :] \
            / float(os * os)
        l = (w // 2 - torch.arange(w, dtype=torch.float64, device=dev)) * pixel + l0
        m = (torch.arange(h, dtype=torch.float64, device=dev) - h // 2) * pixel + m0
        r2 = l[None, :] ** 2 + m[:, None] ** 2
        self.inside = r2 < 1.0
        self.np_ = torch.where(self.inside, torch.sqrt((1.0 - r2).clamp(min=0.0)) - 1.0,
                               torch.zeros_like(r2))
        lo = -max_w if cplx else min_w
        self.layer_w = [0.0] if layers == 1 else \
            [lo + i * (max_w - lo) / (layers - 1) for i in range(layers)]
        u, v, ww = ((uvw[:, i:i + 1] / wl[None, :]).reshape(-1) for i in range(3))
        self.rot = torch.polar(torch.ones_like(u), -2.0 * math.pi * torch.frac(u * l0 + v * m0)) \
            if rotate else None
        self.conj = (ww < 0) & (not cplx)
        sign = torch.where(self.conj, -1.0, 1.0)
        u, v, ww = u * sign, v * sign, ww * sign
        away = lambda t: torch.trunc(t + torch.copysign(torch.full_like(t, 0.5), t))  # noqa: E731
        if layers == 1:
            layer = torch.zeros_like(u)
        else:
            layer = away((ww - lo) * (layers - 1) / (max_w - lo))
        x_exact, y_exact = u * pixel * w, v * pixel * h
        x, y = away(x_exact), away(y_exact)
        self.layer_ok = (layer >= 0) & (layer < layers)
        self.ok = self.layer_ok & (x > -(w // 2)) & (y > -(h // 2)) & (x <= w // 2) & (y <= h // 2)
        self.kx = ((away((x_exact - x) * os).long() + os * 3 // 2) % os)[self.ok]
        self.ky = ((away((y_exact - y) * os).long() + os * 3 // 2) % os)[self.ok]
        self.x, self.y = x.long()[self.ok] - KERNEL // 2, y.long()[self.ok] - KERNEL // 2
        layer = layer.long()[self.ok]
        # by layer, then by footprint, so that the samples of one footprint follow each other
        order = torch.argsort((layer * h + y.long()[self.ok] % h) * w + x.long()[self.ok] % w)
        self.at = torch.nonzero(self.ok).reshape(-1)[order]
        self.kx, self.ky, self.x, self.y = (t[order] for t in (self.kx, self.ky, self.x, self.y))
        self.starts = torch.searchsorted(layer[order].contiguous(),
                                         torch.arange(layers + 1, device=dev)).tolist()

    def _taps(self, a, b):
        for j in range(KERNEL):
            row = torch.remainder(self.y[a:b] + j, self.h) * self.w
            ky = self.tab[self.ky[a:b], j]
            for i in range(KERNEL):
                yield row + torch.remainder(self.x[a:b] + i, self.w), \
                    ky * self.tab[self.kx[a:b], i]

    def _fft_order(self, image, backward):
        """A centred image in the order of the layer's transform."""
        if backward:
            ys = torch.remainder(self.h - torch.arange(self.h, device=self.dev) + self.h // 2,
                                 self.h)
            xs = torch.remainder(torch.arange(self.w, device=self.dev) + self.w // 2, self.w)
        else:
            ys = torch.remainder(torch.arange(self.h, device=self.dev) + self.h // 2, self.h)
            xs = torch.remainder(self.w - torch.arange(self.w, device=self.dev) + self.w // 2,
                                 self.w)
        return ys, xs, image[ys][:, xs]

    def invert(self, vis, factor):
        """vis complex128 [samples] (weighted); real (and imaginary) image."""
        if self.rot is not None:
            vis = vis * self.rot
        vis = torch.where(self.conj, vis.conj(), vis)[self.at]
        total = torch.zeros((self.h, self.w), dtype=torch.complex128, device=self.dev)
        ys, xs, np_ = self._fft_order(self.np_, True)
        for i, w in enumerate(self.layer_w):
            a, b = self.starts[i], self.starts[i + 1]
            if a == b:
                continue
            grid = torch.zeros(self.h * self.w, dtype=torch.complex128, device=self.dev)
            first = torch.remainder(self.y[a:b], self.h) * self.w + \
                torch.remainder(self.x[a:b], self.w)
            _, counts = torch.unique_consecutive(first, return_counts=True)
            last = torch.cumsum(counts, 0) - 1  # of the samples of each footprint
            for cell, k in self._taps(a, b):
                sums = torch.cumsum(vis[a:b] * k, 0)[last]
                sums[1:] -= sums[:-1].clone()
                grid[cell[last]] += sums  # (each cell once)
            f = torch.fft.ifft2(grid.reshape(self.h, self.w), norm="forward")
            total += f * torch.polar(torch.ones_like(np_), -2.0 * math.pi * torch.frac(w * np_))
        out = torch.empty_like(total)
        out[ys[:, None], xs[None, :]] = total
        out = out * factor / self.corr
        return out.real.contiguous(), out.imag.contiguous()

    def predict(self, re, im, nan=True):
        re = re.double()
        model = torch.complex(re, -im.double() if self.cplx else torch.zeros_like(re))
        model = torch.where(self.inside, model, torch.zeros_like(model)) / self.corr
        _, _, model = self._fft_order(model, False)
        _, _, np_ = self._fft_order(self.np_, False)
        out = torch.full((self.ok.numel(),), complex(math.nan, math.nan) if nan else 0.0,
                         dtype=torch.complex128, device=self.dev)
        for i, w in enumerate(self.layer_w):
            a, b = self.starts[i], self.starts[i + 1]
            if a == b:
                continue
            layer = torch.fft.fft2(
                model * torch.polar(torch.ones_like(np_), -2.0 * math.pi * torch.frac(w * np_)))
            layer = layer.reshape(-1)
            acc = torch.zeros(b - a, dtype=torch.complex128, device=self.dev)
            for cell, k in self._taps(a, b):
                acc += layer[cell] * k
            out[self.at[a:b]] = acc
        out = torch.where(self.conj, out, out.conj())
        if self.rot is not None:
            out = out * self.rot.conj()
        return out


def _exact_weights(case, s):
    """Imaging weight of every sample: the weights' grid over the v >= 0 half
    plane, uniform, Briggs (robust 0) or natural."""
    u = (s["uvw"][:, 0:1] / s["wl"][None, :]).reshape(-1)
    v = (s["uvw"][:, 1:2] / s["wl"][None, :]).reshape(-1)
    u, v = torch.where(v < 0, -u, u), v.abs()
    w, h = case["width"], case["height"]
    x = torch.floor(u * w * s["pixel"] + w // 2)
    y = torch.floor(v * h * s["pixel"])
    inside = (x >= 0) & (x < w) & (y < h // 2)
    cell = torch.where(inside, x + y * w, torch.zeros_like(x)).long()
    weight = s["weights"][..., 0].reshape(-1).double() * inside
    order = torch.argsort(cell)
    cells, counts = torch.unique_consecutive(cell[order], return_counts=True)
    last = torch.cumsum(counts, 0) - 1
    sums = torch.cumsum(weight[order], 0)[last]
    sums[1:] -= sums[:-1].clone()
    grid = torch.zeros(w * (h // 2), dtype=torch.float64, device=u.device)
    grid[cells] = sums
    if case["weighting"] == "uniform":
        grid = torch.where(grid != 0, 1.0 / grid, grid)
    elif case["weighting"] == "natural":
        grid = (grid != 0).double()
    else:
        grid = 1.0 / (1.0 + grid * (25.0 * weight.sum() / (grid * grid).sum()))
    return torch.where(inside, grid[cell], torch.zeros_like(weight))


def _exact_direct(case, s):
    dev, pixel, w, h = s["dev"], s["pixel"], case["width"], case["height"]
    l = (w // 2 - torch.arange(w, dtype=torch.float64, device=dev)) * pixel
    m = (torch.arange(h, dtype=torch.float64, device=dev) - h // 2) * pixel
    ll, mm = l[None, :].expand(h, w).reshape(-1), m[:, None].expand(h, w).reshape(-1)
    nn = torch.sqrt(1.0 - ll * ll - mm * mm) - 1.0
    u, v, ww = ((s["uvw"][:, i:i + 1] / s["wl"][None, :]).reshape(-1) for i in range(3))
    vis = s["vis"].reshape(-1).to(torch.complex128)
    img = torch.zeros(w * h, dtype=torch.float64, device=dev)
    step = max(1, (1 << 27) // (w * h))
    for a in range(0, u.numel(), step):
        b = min(u.numel(), a + step)
        turns = u[a:b, None] * ll + v[a:b, None] * mm + ww[a:b, None] * nn
        ph = 2.0 * math.pi * torch.frac(turns)
        img += (vis.real[a:b, None] * torch.cos(ph) + vis.imag[a:b, None] * torch.sin(ph)).sum(0)
    model = s["model"][0].reshape(-1).double()
    at = torch.nonzero(model).reshape(-1)
    out = torch.zeros(u.numel(), dtype=torch.complex128, device=dev)
    for a in range(0, u.numel(), 1 << 18):
        b = min(u.numel(), a + (1 << 18))
        turns = u[a:b, None] * ll[at] + v[a:b, None] * mm[at] + ww[a:b, None] * nn[at]
        ph = torch.polar(torch.ones_like(turns), 2.0 * math.pi * torch.frac(turns))
        out[a:b] = ph @ model[at].to(torch.complex128)
    return {"image": img.reshape(h, w) * _factor(s), "vis": out.reshape(-1, case["channels"])}


def exact(case, seed):
    rows, nchan = _samples(case)
    n, op = case["images"], case["op"]
    ways = 1 if op in ("invert", "predict") else 2
    facets = max(1, case["facets"])
    layers = case["layers"] or 30
    # seconds: taps, transforms
    if op != "direct" and ways * facets * n * (
            rows * nchan * KERNEL * KERNEL / 2e9 +
            layers * case["width"] * case["height"] * 1.5e-9) > 12.0:
        return None
    s = _inputs(case, seed)
    if op == "direct":
        return _exact_direct(case, s)
    cplx = _complex(case)
    shape = (rows, nchan)
    if op == "facets":
        from wsclean_amd.autotune import suggested_w_layers
        min_w = float(s["uvw"][:, 2].abs().min() / s["wl"].max())
        max_w = float(s["uvw"][:, 2].abs().max() / s["wl"].min())
        re, im, vis = [], [], []
        for i, f in enumerate(s["facets"]):
            nw = suggested_w_layers(f.box[2] - f.box[0], f.box[3] - f.box[1], FACET_PIXEL,
                                    FACET_PIXEL, -max_w if cplx else min_w, max_w, f.l_shift,
                                    f.m_shift)
            kinds = [_Exact(f.width, f.height, FACET_PIXEL, nw, min_w, max_w,
                            case["oversampling"], c, s["uvw"], s["wl"], f.l_shift, f.m_shift,
                            True) for c in ((False, True) if cplx else (False,))]
            got = [kinds[1 if j in cplx else 0].invert(
                s["vis"][..., j].reshape(-1).to(torch.complex128), 1.0 / (rows * nchan))
                for j in range(n)]
            re.append(torch.stack([g[0] for g in got]))
            if cplx:
                im.append(torch.stack([g[1] if j in cplx else torch.zeros_like(g[1])
                                       for j, g in enumerate(got)]))
            vis.append(torch.stack([kinds[1 if j in cplx else 0].predict(
                s["model"][i][j], s["model_im"][i][j] if cplx else None).reshape(shape)
                for j in range(n)], dim=-1))
        return {"re": re, "im": im if cplx else None, "vis": vis}
    kinds = [_Exact(case["width"], case["height"], s["pixel"], case["layers"], s["min_w"],
                    s["max_w"], case["oversampling"], c, s["uvw"], s["wl"])
             for c in ((False, True) if cplx else (False,))]
    if op == "grad":
        vis = kinds[0].predict(s["model"][0], None, nan=False)
        d = vis - s["vis"].reshape(-1).to(torch.complex128)
        grad, _ = kinds[0].invert(2.0 * d, 1.0)
        return {"vis": vis.reshape(shape), "loss": (d.abs() ** 2).sum(), "grad": grad}
    got = {}
    if op != "predict":
        imgw = _exact_weights(case, s) if case["weighting"] != "none" else None
        images = []
        for j in range(n):
            k = kinds[1 if j in cplx else 0]
            v, factor = s["vis"][..., j].reshape(-1).to(torch.complex128), _factor(s)
            if imgw is not None:
                cw = imgw * s["weights"][..., j].reshape(-1).double()
                v, factor = v * cw, factor / float(cw[k.layer_ok].sum())
            images.append(k.invert(v, factor))
        re = torch.stack([g[0] for g in images])
        if op == "host":
            got["image"] = re
        else:
            got["re"] = re
            got["im"] = torch.stack([g[1] if j in cplx else torch.zeros_like(g[1])
                                     for j, g in enumerate(images)]) if cplx else None
    if op != "invert":
        vis = torch.stack([kinds[1 if j in cplx else 0].predict(
            s["model"][j], s["model_im"][j] if cplx else None).reshape(shape)
            for j in range(n)], dim=-1)
        got["vis"] = vis
    return got
