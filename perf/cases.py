"""Performance cases of the imaging and source-finding path.

Each case is one pass a program makes through the public entry points: imaging of
one snapshot on device buffers (with and without W-projection), of a batch of
snapshots, of host arrays; source finding on an image; a whole snapshot; model
visibilities.  The sizes are those of the repository's benchmark workloads and of
the configurations under tests/golden/configs, with odd visibility counts and image
shapes beside them.

Two uv coverages are used: "disk" (uniform in a disk of radius 0.45 / cell, the
benchmark workloads' recipe) and "array" (the baselines of a centrally condensed
array over several channels: most visibilities near the origin of the uv plane, as
interferometers measure them).
"""
import ctypes
import math
import weakref

import numpy as np
import torch

from fastimaging_amd import capi
from fastimaging_amd.stp import Context

ARCSEC = math.pi / (180.0 * 3600.0)
KERNELS = {"gaussiansinc": capi.KERNEL_GAUSSIANSINC, "pswf": capi.KERNEL_PSWF, "gaussian": capi.KERNEL_GAUSSIAN}
MEDIANS = {"binmedian": capi.MEDIAN_BINMEDIAN, "binapprox": capi.MEDIAN_BINAPPROX}
PRECISIONS = {"f64": capi.PRECISION_FP64, "f32": capi.PRECISION_FP32C}
DTYPES = {"f64": torch.float64, "f32": torch.float32}
ISLAND_CAPACITY = 1 << 17

IMAGE = dict(op="image", size=4096, padding=1, cell=1.0, n_vis=1_000_000, sources=50, uv="disk", w_max=0.0,
             kernel="gaussiansinc", support=3, exact=False, oversampling=8, beam=True, gcf=False, analytic_gcf=False,
             planes=0, w_support=0, trunc=0.0, precision="f32")
FIND = dict(op="find", rows=4096, cols=4096, precision="f32", beam_px=1.2, sources=50, detection=5.0, analysis=3.0,
            median="binmedian", conn4=False, negative=True)


def listed():
    return [
        # the smallest call: a few baselines' worth of host arrays through the drop-in entry point
        dict(IMAGE, name="host-256-f64", op="host", size=256, n_vis=2_000, sources=3, precision="f64"),
        # a small snapshot through the whole pipeline, launch latency above all
        dict(IMAGE, name="snapshot-1024-f64", op="snapshot", size=1024, n_vis=50_000, sources=5, precision="f64",
             oversampling=9, beam_px=1.2, detection=5.0, analysis=3.0, median="binmedian", conn4=False, negative=True),
        # exact PSWF kernels, padded and grid-corrected (the exact-PSWF configuration)
        dict(IMAGE, name="image-1024-pswf-exact-f64", size=1024, padding=2, cell=0.5, n_vis=300_001, sources=10,
             uv="array", kernel="pswf", exact=True, oversampling=1, gcf=True, analytic_gcf=True, precision="f64"),
        # the headline snapshot's imaging
        dict(IMAGE, name="image-4096-f32", oversampling=9),
        # the same size in double precision with an array's uv coverage, ragged count
        dict(IMAGE, name="image-4096-array-f64", n_vis=1_000_003, uv="array", precision="f64"),
        # the largest snapshots: PSWF, grid-corrected, no beam (the simple configuration)
        dict(IMAGE, name="image-8192-f32", size=8192, cell=0.5, n_vis=4_000_000, sources=20, uv="array", kernel="pswf",
             beam=False, gcf=True, analytic_gcf=True),
        # wide-field imaging, the W-projection benchmark workload
        dict(IMAGE, name="wproj-4096-f32", cell=2.0, n_vis=2_000_000, sources=40, w_max=1500.0, planes=32, w_support=32),
        # W-projection as configured for wide fields: truncated Gaussian kernels, grid correction, no beam
        dict(IMAGE, name="wproj-2048-trunc-f64", size=2048, cell=60.0, n_vis=300_007, sources=10, uv="array",
             w_max=100.0, kernel="gaussian", beam=False, gcf=True, analytic_gcf=True, planes=24, w_support=31,
             trunc=1.0, precision="f64"),
        # a batch of snapshots of mixed sizes, imaging only
        dict(IMAGE, name="batch-12-f32", op="batch", count=12, n_min=20_000, n_max=2_000_000, oversampling=9),
        # source finding on a headline-sized image, islands to host
        dict(FIND, name="find-4096-f32"),
        # source finding on an odd-shaped image, well-sampled beam, the library's default median
        dict(FIND, name="find-3000x2600-f64", rows=3000, cols=2600, precision="f64", beam_px=3.5, sources=200,
             detection=4.5, analysis=3.0, median="binapprox", conn4=True),
        # the model visibilities of a local sky model, one for each measured visibility
        dict(op="model", name="model-1M-50", n_vis=1_000_000, sources=50, cell=1.0, size=4096, uv="disk",
             w_max=1500.0),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["image", "image", "image", "wproj", "batch", "find", "find", "snapshot", "host", "model"])
    if op == "model":
        return dict(op="model", n_vis=_log(rng, 1e4, 2e6), sources=rng.randint(1, 50), cell=1.0, size=4096,
                    uv=rng.choice(["disk", "array"]), w_max=rng.choice([0.0, 1500.0]))
    if op == "find":
        return dict(FIND, rows=2 * _log(rng, 128, 2048), cols=2 * _log(rng, 128, 2048),
                    precision=rng.choice(["f32", "f64"]), beam_px=round(rng.uniform(1.2, 4.0), 2),
                    sources=rng.randint(1, 300), detection=rng.choice([4.5, 5.0, 20.0]),
                    analysis=rng.choice([3.0, 4.0]), median=rng.choice(["binmedian", "binapprox"]),
                    conn4=rng.random() < 0.3, negative=rng.random() < 0.7)
    kernel, gcf, analytic = rng.choice([("gaussiansinc", False, False), ("gaussiansinc", True, False),
                                        ("pswf", True, True), ("gaussian", True, True)])
    case = dict(IMAGE, op=op, kernel=kernel, gcf=gcf, analytic_gcf=analytic, sources=rng.randint(1, 40),
                uv=rng.choice(["disk", "array"]), beam=rng.random() < 0.7, precision=rng.choice(["f64", "f32"]),
                oversampling=rng.choice([4, 8, 9]), support=rng.choice([3, 3, 3, 5, 7]))
    if op == "wproj":
        w_support = rng.randint(8, 32)
        case.update(op="image", size=rng.choice([1024, 2048, 4096]), cell=2.0, n_vis=_log(rng, 2e4, 2e6), w_max=1500.0,
                    planes=rng.randint(4, 32), w_support=w_support, trunc=rng.choice([0.0, 1.0]), support=3,
                    oversampling=8)
    elif op == "batch":
        case.update(count=rng.randint(3, 12), n_min=10_000, n_max=rng.choice([200_000, 2_000_000]), beam=True,
                    gcf=False, analytic_gcf=False, kernel="gaussiansinc")
    elif op in ("host", "snapshot"):
        case.update(size=rng.choice([256, 512, 1024]), n_vis=_log(rng, 1e3, 1e5), precision="f64")
    else:
        size = rng.choice([512, 1024, 2048, 4096, 8192])
        padding = rng.choice([1, 1, 2]) if size < 8192 else 1
        exact = rng.random() < 0.2
        case.update(size=size, padding=padding, n_vis=_log(rng, 1e4, 4e6 if not exact else 1e6), exact=exact)
        if exact:
            case["oversampling"] = 1
    if op == "snapshot":
        case.update(beam_px=1.2, detection=5.0, analysis=3.0, median=rng.choice(["binmedian", "binapprox"]),
                    conn4=rng.random() < 0.3, negative=True)
    return case


# ---------------------------------------------------------------- inputs
_context = None


def _ctx():
    """The handle a program keeps for all of its calls."""
    global _context
    if _context is None:
        _context = Context(0)
    return _context


def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _uniform(g, *shape):
    return torch.rand(*shape, generator=g, device="cuda", dtype=torch.float64)


def _normal(g, *shape):
    return torch.randn(*shape, generator=g, device="cuda", dtype=torch.float64)


def _uvw(g, n, uv, cell, w_max):
    """(3, n): the columns u, v, w in wavelengths."""
    radius = 0.45 / (cell * ARCSEC)
    out = torch.zeros(3, n, device="cuda", dtype=torch.float64)
    if uv == "disk":
        r = radius * torch.sqrt(_uniform(g, n))
        phi = 2.0 * math.pi * _uniform(g, n)
        out[0], out[1] = r * torch.cos(phi), r * torch.sin(phi)
        if w_max > 0.0:
            out[2] = (2.0 * _uniform(g, n) - 1.0) * w_max
        return out
    # an array of antennas, denser towards its centre, all baselines over some channels
    channels = 8
    ants = max(4, int(math.ceil(0.5 + math.sqrt(0.25 + 2.0 * n / channels))))
    r = 0.5 * _uniform(g, ants) ** 1.5
    phi = 2.0 * math.pi * _uniform(g, ants)
    pos = torch.stack([r * torch.cos(phi), r * torch.sin(phi)])
    a, b = torch.triu_indices(ants, ants, offset=1, device="cuda")
    base = pos[:, a] - pos[:, b]
    scale = 0.8 + 0.2 * torch.arange(1, channels + 1, device="cuda", dtype=torch.float64) / channels
    uv2 = (base[:, None, :] * scale[None, :, None]).reshape(2, -1)[:, :n]
    out[0], out[1] = radius * uv2[0], radius * uv2[1]
    if w_max > 0.0:  # a plane array seen at an angle, with some height differences
        out[2] = w_max * (0.6 * uv2[0] + 0.3 * uv2[1] + 0.1 * (2.0 * _uniform(g, n) - 1.0))
    return out


def _skymodel(g, sources, size, cell):
    half = 0.25 * size * cell * ARCSEC
    lm = (2.0 * _uniform(g, 2, sources) - 1.0) * half
    flux = 0.5 * torch.exp(_uniform(g, sources) * math.log(40.0))
    return lm[0], lm[1], flux


def _model(uvw, sky, sign):
    """sum_k A_k exp(sign 2 pi i (u l + v m + w (n - 1)))."""
    out = torch.zeros(uvw.shape[1], device="cuda", dtype=torch.complex128)
    for l, m, a in zip(*(x.tolist() for x in sky)):
        ph = uvw[0] * l + uvw[1] * m + uvw[2] * (math.sqrt(1.0 - l * l - m * m) - 1.0)
        out += torch.polar(torch.full_like(ph, a), sign * 2.0 * math.pi * ph)
    return out


def _snapshot(g, n, case):
    uvw = _uvw(g, n, case["uv"], case["cell"], case["w_max"])
    vis = _model(uvw, _skymodel(g, case["sources"], case["size"], case["cell"]), -1.0)
    vis += 0.1 * torch.complex(_normal(g, n), _normal(g, n))
    weights = 0.5 + _uniform(g, n)
    return dict(uvw=uvw, vis=vis, weights=weights)


def _batch(case):
    """(image size, visibilities) of a batch's snapshots; the sizes belong to the case."""
    sizes = np.random.RandomState(1000 + case["count"])
    out = []
    for _ in range(case["count"]):
        N = 2048 if sizes.rand() < 0.5 else 4096
        n = int(round(math.exp(sizes.uniform(math.log(case["n_min"]), math.log(case["n_max"])))))
        out.append((N, n))
    return out


def _sky_image(g, case):
    """Noise and sources at the resolution of the beam, in the imager's un-shifted layout."""
    rows, cols = case["rows"], case["cols"]
    fy = torch.fft.rfftfreq(rows, device="cuda", dtype=torch.float64)
    fx = torch.fft.fftfreq(cols, device="cuda", dtype=torch.float64)
    f2 = fx[:, None] ** 2 + fy[None, :] ** 2
    beam = torch.exp(-(math.pi * case["beam_px"]) ** 2 / (4.0 * math.log(2.0)) * f2)
    noise = torch.fft.irfftn(torch.fft.rfftn(_normal(g, cols, rows)) * beam, s=(cols, rows))
    noise *= 0.02 / noise.std()
    img = torch.zeros(cols, rows, device="cuda", dtype=torch.float64)
    k = case["sources"]
    x = (_uniform(g, k) * cols).long().clamp(max=cols - 1)
    y = (_uniform(g, k) * rows).long().clamp(max=rows - 1)
    img[x, y] = 0.1 * torch.exp(_uniform(g, k) * math.log(100.0))
    img = torch.fft.irfftn(torch.fft.rfftn(img) * beam, s=(cols, rows))
    img *= (math.pi * case["beam_px"] ** 2) / (4.0 * math.log(2.0))
    return (img + noise).to(DTYPES[case["precision"]]).contiguous()


def _imager_pars(case, size=None):
    size = size or case["size"]
    return capi.imager_pars(size, case["cell"], kernel_function=KERNELS[case["kernel"]],
                            kernel_support=case["support"], kernel_exact=case["exact"],
                            oversampling=case["oversampling"], generate_beam=case["beam"],
                            gridding_correction=case["gcf"], analytic_gcf=case["analytic_gcf"],
                            padding_factor=float(case["padding"]))


def _find_pars(case):
    return capi.sourcefind_pars(case["detection"], case["analysis"], find_negative_sources=case["negative"],
                                median_method=MEDIANS[case["median"]], ccl_4connectivity=case["conn4"])


class _Find:
    """What a program keeps for source finding: its label map and a page-locked island list."""

    def __init__(self, case, rows, cols):
        self.ctx = _ctx()
        self.pars = _find_pars(case)
        self.rows, self.cols = rows, cols
        self.labels = torch.empty(cols, rows, device="cuda", dtype=torch.int32)
        self.islands = self.ctx.island_buffer(ISLAND_CAPACITY)
        ctypes.memset(self.islands, 0, ctypes.sizeof(self.islands))
        # given back when the last view of it is gone
        weakref.finalize(self.islands, self.ctx.lib.stp_host_free, self.ctx.h, self.islands._stp_host_ptr)

    def run(self, image, precision):
        _, st = self.ctx.source_find_device(image.data_ptr(), self.rows, self.cols, self.pars,
                                            d_label_map=self.labels.data_ptr(), precision=precision, out=self.islands)
        # the records as the library wrote them; those past the last island are zero
        words = np.frombuffer(self.islands, dtype=np.int32).reshape(-1, 24)
        reals = np.frombuffer(self.islands, dtype=np.float64).reshape(-1, 12)
        return dict(label_map=self.labels, island_ints=words[:, :5], extremum=reals[:, 3], position=reals[:, 6:9],
                    semimajor=reals[:, 9], bg_level=st.bg_level, rms_est=st.rms_est, mean=st.mean, sigma=st.sigma,
                    counts=[st.num_labels_pos, st.num_labels_neg, st.num_valid_labels, st.num_islands])


def prepare(case, seed):
    g = _generator(seed)
    op, ctx = case["op"], _ctx()
    s = dict(op=op, ctx=ctx)
    if op == "model":
        s["uvw"] = _uvw(g, case["n_vis"], case["uv"], case["cell"], case["w_max"])
        sky = _skymodel(g, case["sources"], case["size"], case["cell"])
        s["vis"] = torch.empty(case["n_vis"], device="cuda", dtype=torch.complex128)
        s["sky"] = np.asfortranarray(torch.stack(sky, 1).cpu().numpy())
        s["n"] = case["n_vis"]
        return s
    s["precision"] = PRECISIONS[case["precision"]]
    if op == "find":
        s["image"] = _sky_image(g, case)
        s["find"] = _Find(case, case["rows"], case["cols"])
        return s
    s["pars"] = _imager_pars(case)
    dtype = DTYPES[case["precision"]]
    if op == "batch":
        s["keep"], s["items"] = [], []
        for N, n in _batch(case):
            snap = _snapshot(g, n, dict(case, size=N))
            image, beam = (torch.empty(N, N, device="cuda", dtype=dtype) for _ in range(2))
            it = capi.BatchItem()
            it.img_pars = _imager_pars(case, N)
            it.n_vis = n
            it.d_vis, it.d_vis_weights, it.d_uvw_lambda, it.d_image, it.d_beam = (
                t.data_ptr() for t in (snap["vis"], snap["weights"], snap["uvw"], image, beam))
            s["items"].append(it)
            s["keep"].append((snap, image, beam))
        return s
    s["wproj"] = capi.wproj_pars(case["planes"], case["w_support"], kernel_trunc_perc=case["trunc"]) \
        if case["planes"] else None
    s.update(_snapshot(g, case["n_vis"], case))
    s["n"] = case["n_vis"]
    if op == "host":
        s["vis"], s["weights"] = s["vis"].cpu().numpy(), s["weights"].cpu().numpy()
        s["uvw"] = s["uvw"].cpu().numpy().T  # (n, 3), column-major
        return s
    s["image"] = torch.empty(case["size"], case["size"], device="cuda", dtype=dtype)
    s["beam"] = torch.empty(case["size"], case["size"], device="cuda", dtype=dtype) if case["beam"] else None
    if op == "snapshot":
        s["find"] = _Find(case, case["size"], case["size"])
    return s


def run(s):
    op, ctx = s["op"], s["ctx"]
    if op == "model":
        ctx.model_visibilities_device(s["sky"], s["n"], s["uvw"].data_ptr(), s["vis"].data_ptr(), subtract=False)
        return s["vis"]
    if op == "find":
        return s["find"].run(s["image"], s["precision"])
    if op == "batch":
        totals = ctx.image_batch(s["items"], precision=s["precision"], flags=capi.BATCH_FUSED)
        return dict(totals=totals, images=[k[1] for k in s["keep"]], beams=[k[2] for k in s["keep"]])
    if op == "host":
        image, beam = ctx.image_visibilities(s["vis"], s["weights"], s["uvw"], s["pars"], w_proj=s["wproj"],
                                             precision=s["precision"])
        return dict(image=image.T, beam=beam.T) if beam is not None else dict(image=image.T)
    ctx.image_visibilities_device(s["pars"], s["n"], s["vis"].data_ptr(), s["weights"].data_ptr(),
                                  s["uvw"].data_ptr(), s["image"].data_ptr(),
                                  s["beam"].data_ptr() if s["beam"] is not None else None, precision=s["precision"],
                                  w_proj=s["wproj"])
    out = dict(image=s["image"])
    if s["beam"] is not None:
        out["beam"] = s["beam"]
    if op == "snapshot":
        out.update(s["find"].run(s["image"], s["precision"]))
    return out


def _imaging_work(case, size, n):
    padded = size * case["padding"]
    real = 8 if case["precision"] == "f64" else 4
    maps = 2 if case["beam"] else 1
    taps = (2 * (case["w_support"] if case["planes"] else case["support"]) + 1) ** 2
    per_tap = (8 if case["planes"] else 4) + ((4 if case["planes"] else 2) if case["beam"] else 0)
    return dict(bytes=48.0 * n + maps * size * size * real,
                flops=1.0 * n * taps * per_tap + maps * 5.0 * padded * padded * math.log2(padded))


def work(case):
    op = case["op"]
    if op == "model":
        # uvw in, visibilities out; a phase, a sine and a cosine per source and visibility
        return dict(bytes=40.0 * case["n_vis"], flops=50.0 * case["n_vis"] * case["sources"])
    if op == "find":
        px = case["rows"] * case["cols"]
        return dict(bytes=px * ((8.0 if case["precision"] == "f64" else 4.0) + 4.0), flops=20.0 * px)
    if op == "batch":
        parts = [_imaging_work(case, N, n) for N, n in _batch(case)]
        return {k: sum(p[k] for p in parts) for k in ("bytes", "flops")}
    out = _imaging_work(case, case["size"], case["n_vis"])
    if op == "snapshot":
        px = case["size"] ** 2
        out["bytes"] += 4.0 * px
        out["flops"] += 20.0 * px
    return out


# ---------------------------------------------------------------- the same in 64 bits, plain torch
def _grdsf(nu):
    p = ((8.203343e-2, -3.644705e-1, 6.278660e-1, -5.335581e-1, 2.312756e-1),
         (4.028559e-3, -3.697768e-2, 1.021332e-1, -1.201436e-1, 6.412774e-2))
    q = ((1.0, 8.212018e-1, 2.078043e-1), (1.0, 9.599102e-1, 2.918724e-1))
    nu = nu.abs()
    parts = []
    for k, end in ((0, 0.75), (1, 1.0)):
        d = nu * nu - end * end
        parts.append(sum(c * d ** i for i, c in enumerate(p[k])) / sum(c * d ** i for i, c in enumerate(q[k])))
    return torch.where(nu < 0.75, parts[0], torch.where(nu <= 1.0, parts[1], torch.zeros_like(nu)))


def _kernel(case, x):
    name, half = case["kernel"], float(case["support"])
    if name == "pswf":
        nu = x / half
        v = _grdsf(nu) * (1.0 - nu * nu)
    else:
        gauss = torch.exp(-(x * x) / (2.52 ** 2 if name == "gaussiansinc" else 1.0))
        v = gauss * torch.sinc(x / 1.55) if name == "gaussiansinc" else gauss
    return torch.where(x.abs() > half, torch.zeros_like(v), v)


def _image_domain(case, size):
    """The kernel's transform over an image of `size` pixels, centred."""
    i = torch.arange(size, device="cuda", dtype=torch.float64) - size // 2
    if case["analytic_gcf"]:
        r = i / (size // 2)
        return _grdsf(r) if case["kernel"] == "pswf" else torch.exp(-(r * math.pi / 2.0) ** 2)
    k = _kernel(case, i)
    k = k / k.sum()
    c = size // 2
    f = torch.fft.fft(torch.cat([k[c:], k[:c]])).real
    return torch.cat([f[c:], f[:c]])


def _w_kernels(case, w_planes, oversampling):
    """(planes, cp_y, cp_x, row, column) convolution kernels."""
    sup, os = case["w_support"], oversampling
    ks, workarea = 2 * sup + 1, 2
    while workarea < ks:
        workarea *= 2
    padded = case["size"] * case["padding"]
    cell = case["cell"] * ARCSEC * (padded / workarea)
    aa = _image_domain(case, workarea)
    half, arr = workarea // 2, workarea * os
    i = torch.arange(half, device="cuda", dtype=torch.float64)
    r2 = (i[:, None] * cell) ** 2 + (i[None, :] * cell) ** 2
    nn = torch.sqrt((1.0 - r2).clamp(min=1e-300))
    taper = aa[half:, None] * aa[None, half:]
    cs, cache = 2 * (os // 2) + 1, []
    for w in w_planes:
        ph = -2.0 * math.pi * w * (nn - 1.0)
        quad = torch.where(r2 >= 1.0, taper.to(torch.complex128), torch.polar(1.0 / nn, ph) * taper)
        quad[0, 0] = taper[0, 0]
        full = torch.zeros(arr, arr, device="cuda", dtype=torch.complex128)
        full[:half, :half] = quad
        full[arr - half + 1:, :half] = quad[1:].flip(0)
        full[:half, arr - half + 1:] = quad[:, 1:].flip(1)
        full[arr - half + 1:, arr - half + 1:] = quad[1:, 1:].flip(0, 1)
        conv = torch.fft.fft2(full)
        s = sup
        if case["trunc"] > 0.0:
            col = conv[:, 0].abs().cpu().numpy()
            k = min(sup * os, arr // 2)
            while k > 0 and not col[k] > col[0] * case["trunc"] / 100.0:
                k -= os
            s = max(1, min(k // os, sup))
        out = torch.zeros(cs, cs, ks, ks, device="cuda", dtype=torch.complex128)
        t = torch.arange(-s, s + 1, device="cuda")
        for y in range(cs):
            rows = (t * os + os // 2 - y) % arr
            for x in range(cs):
                cut = conv[rows][:, (t * os + os // 2 - x) % arr]
                out[y, x, sup - s:sup + s + 1, sup - s:sup + s + 1] = cut / cut.real.sum()
        cache.append(out)
    return torch.stack(cache)


def _exact_image(case, snap):
    N = case["size"] * case["padding"]
    half, rows = N // 2, N // 2 + 1
    wproj, exact = case["planes"] > 0, case["exact"]
    sup = case["w_support"] if wproj else case["support"]
    os = 1 if exact else max(1, case["oversampling"] // 2 * 2)
    px = (case["cell"] / 3600.0) * (math.pi / 180.0) * N
    u, v, w = snap["uvw"][0] * px, snap["uvw"][1] * px, snap["uvw"][2].clone()
    vis, wt = snap["vis"].clone(), snap["weights"]
    if wproj:
        order = torch.sort(w.abs(), stable=True).indices
        u, v, w, vis, wt = u[order], v[order], w[order], vis[order], wt[order]
    neg = v < 0.0
    twice = v.abs() < sup + 1
    flip = torch.where(neg, -1.0, 1.0).to(torch.float64)
    u, v, w = u * flip, v * flip, w * flip
    vis = torch.where(neg, vis.conj(), vis)
    cx, cy = torch.round(u), torch.round(v)
    fx, fy = u - cx, v - cy
    cx, cy = cx.long() + half, cy.long() + half
    good = (cx - sup > 0) & (cy - sup > 0) & (cx + sup < N) & (cy + sup < N)
    cx, cy = torch.where(cx < half, cx + half, cx - half), torch.where(cy < half, cy + half, cy - half)
    total = 2.0 * float(wt[good].sum())
    plane = torch.zeros_like(cx)
    means = []
    if wproj:
        g = good.cpu().numpy()
        cum, aw = np.cumsum(g), w.abs().cpu().numpy()
        begin = 0
        for k in range(case["planes"]):
            size = int(math.ceil((int(cum[-1]) - begin) / (case["planes"] - k)))
            before = int(cum[begin - 1]) if begin else 0
            end = min(len(g), int(np.searchsorted(cum, before + size)) + 1) if size > 0 else begin
            sel = g[begin:end]
            means.append(float(aw[begin:end][sel].mean()) if sel.any() else 0.0)
            plane[begin:end if k < case["planes"] - 1 else len(g)] = k
            begin = end
    # the copies of visibilities near v = 0, conjugated, at the mirrored position
    lim = os // 2
    ox = (torch.round(fx * os).long().clamp(-lim, lim) + lim)
    oy = (torch.round(fy * os).long().clamp(-lim, lim) + lim)
    a, b = good, good & twice
    cat = lambda p, q: torch.cat([p[a], q[b]])  # noqa: E731
    X, Y = cat(cx, N - cx), cat(cy, N - cy)
    OX, OY = (cat(ox, os - ox), cat(oy, os - oy)) if os > 1 else (cat(ox, ox), cat(oy, oy))
    FX, FY = cat(fx, -fx), cat(fy, -fy)
    V, W, T, P = cat(vis, vis.conj()), cat(w, -w), cat(wt, wt), cat(plane, plane)
    maps = 2 if case["beam"] else 1
    grid = torch.zeros(maps, N * rows, 2, device="cuda", dtype=torch.float64)
    if wproj:
        cache = _w_kernels(case, means, os)
        cs, ks = 2 * (os // 2) + 1, 2 * sup + 1
        sub = (P * cs + OY) * cs + OX
        cache = cache.reshape(-1, ks, ks).permute(1, 2, 0).contiguous()
        sign = torch.where(W < 0.0, -1.0, 1.0).to(torch.float64)
    else:
        t = torch.arange(-sup, sup + 1, device="cuda", dtype=torch.float64)
        offx, offy = (FX, FY) if exact else ((OX - lim).double() / os, (OY - lim).double() / os)
        kx, ky = _kernel(case, t[None, :] - offx[:, None]), _kernel(case, t[None, :] - offy[:, None])
        kx, ky = kx / kx.sum(1, keepdim=True), ky / ky.sum(1, keepdim=True)
    for i in range(2 * sup + 1):
        r = Y - sup + i
        r = torch.where(r >= N, r - N, r)
        inside = torch.nonzero((r >= 0) & (r < rows)).reshape(-1)
        r, x, vv, tt = r[inside], X[inside], V[inside], T[inside]
        for j in range(2 * sup + 1):
            if wproj:
                k = cache[i, j][sub[inside]]
                k = torch.complex(k.real, k.imag * sign[inside]) * tt
            else:
                k = (kx[inside, j] * ky[inside, i] * tt).to(torch.complex128)
            at = ((x - sup + j) % N) * rows + r
            grid[0].index_add_(0, at, torch.view_as_real(vv * k))
            if maps == 2:
                grid[1].index_add_(0, at, torch.view_as_real(k))
    out = []
    keep = torch.cat([torch.arange(case["size"] // 2), torch.arange(N - case["size"] // 2, N)]).cuda()
    corr = _image_domain(case, N).roll(-half)[keep] if case["gcf"] else None
    for k in range(maps):
        f = torch.fft.ifft(torch.view_as_complex(grid[k]).reshape(N, rows), dim=0, norm="forward")
        f[:, 0].imag.zero_()
        f[:, -1].imag.zero_()
        img = torch.fft.irfft(f, n=N, dim=1, norm="forward")[keep][:, keep] / total
        out.append(img / (corr[:, None] * corr[None, :]) if corr is not None else img)
    return (out[0], out[1] if maps == 2 else None, total)


def _components(cls, conn4):
    """First scan position of each pixel's component; cls (cols, rows) of the visual image."""
    cols, rows = cls.shape
    big = cols * rows
    r = (torch.arange(rows, device="cuda") + rows // 2) % rows
    key = torch.arange(cols, device="cuda")[:, None] * rows + r[None, :]
    key = torch.where(cls != 0, key, big)
    pad = torch.nn.functional.pad
    c = pad(cls, (1, 1, 1, 1))
    steps = [(0, 1), (1, 0), (0, -1), (-1, 0)] + ([] if conn4 else [(1, 1), (1, -1), (-1, 1), (-1, -1)])
    while True:
        k, new = pad(key, (1, 1, 1, 1), value=big), key
        for dx, dy in steps:
            near = (slice(1 + dx, 1 + dx + cols), slice(1 + dy, 1 + dy + rows))
            new = torch.where((c[near] == cls) & (cls != 0), torch.minimum(new, k[near]), new)
        if torch.equal(new, key):
            return key
        key = new


def _exact_find(case, image):
    cols, rows = image.shape
    x = image.double().reshape(-1)
    n = x.numel()
    mean = float(x.mean())
    sigma = float(torch.sqrt((x * x).mean() - mean * mean))
    if case["median"] == "binapprox" and 2.0 * sigma >= 0.0001:
        scale, left = 1000 / (2.0 * sigma), mean - sigma
        b = ((x - left) * scale).trunc()
        count = int((b < 0).sum())
        bins = torch.bincount(b[(b >= 0) & (b <= 1000)].long(), minlength=1001).cpu().numpy()
        i = int(np.searchsorted(count + np.cumsum(bins), n // 2))
        j, count = i, count + int(bins[:i + 1].sum())
        while count == n // 2 and j < 1000:
            j += 1
            count += int(bins[j])
        bg = (i + j + 1) / (2.0 * scale) + left
    else:
        top = torch.sort(x).values
        bg = float(top[n // 2 - 1] + top[n // 2]) / 2.0
    d = x - bg
    rms, left = sigma, d
    for _ in range(5):
        kept = left[left.abs() <= 3.0 * rms]
        if kept.numel() == left.numel():
            break
        left = kept
        rms = float(torch.sqrt((left * left).mean() - left.mean() ** 2))
    img = image.double().roll((cols // 2, rows // 2), (0, 1))
    cls = (img > bg + case["analysis"] * rms).long()
    if case["negative"]:
        cls -= (img < bg - case["analysis"] * rms).long()
    at = torch.nonzero(cls)
    key = _components(cls, case["conn4"])[at[:, 0], at[:, 1]]
    val, sgn = img[at[:, 0], at[:, 1]], cls[at[:, 0], at[:, 1]]
    out = []
    for s in (1, -1):
        m = sgn == s
        _, lab = torch.unique(key[m], return_inverse=True)
        v, px, py = val[m], at[m][:, 0].double(), at[m][:, 1].double()
        k = int(lab.max()) + 1 if lab.numel() else 0
        add = lambda q: torch.zeros(k, device="cuda", dtype=torch.float64).index_add_(0, lab, q)  # noqa: E731,B023
        ext = s * torch.zeros(k, device="cuda", dtype=torch.float64).scatter_reduce_(0, lab, s * v, "amax", include_self=False)
        flux = add(v)
        xb, yb = add(px * v) / flux, add(py * v) / flux
        dx, dy = px - xb[lab], py - yb[lab]
        xx, yy, xy = add(dx * dx * v) / flux, add(dy * dy * v) / flux, add(dx * dy * v) / flux
        major = (xx + yy) / 2.0 + torch.sqrt((xx - yy) ** 2 / 4.0 + xy * xy)
        ratio = s * ext / (case["analysis"] * rms)
        major = torch.sqrt(major / (1.0 - torch.log(ratio) / (ratio - 1.0)))
        ok = (add(torch.ones_like(v)) >= 5) & (s * ext > s * (bg + s * case["detection"] * rms))
        out.append(torch.stack([ext, ext, xb, yb, major])[:, ok])
    f = torch.cat(out, 1)
    f = torch.nn.functional.pad(f, (0, ISLAND_CAPACITY - f.shape[1]))
    return dict(label_map=None, island_ints=None, extremum=f[0], position=f[1:4].T.contiguous(), semimajor=f[4],
                bg_level=float(bg), rms_est=rms, mean=mean, sigma=sigma, counts=[None] * 4)


def exact(case, seed):
    s = prepare(case, seed)
    op = case["op"]
    if op == "model":
        sky = [torch.from_numpy(s["sky"][:, k].copy()) for k in range(3)]
        scale = torch.sqrt(1.0 - sky[0] ** 2 - sky[1] ** 2)
        return _model(s["uvw"], (sky[0], sky[1], sky[2] * scale), 1.0)
    if op == "find":
        return _exact_find(case, s["image"])
    if op == "batch":
        parts = [_exact_image(dict(case, size=N), k[0]) for (N, n), k in zip(_batch(case), s["keep"])]
        return dict(totals=np.array([p[2] for p in parts]), images=[p[0] for p in parts], beams=[p[1] for p in parts])
    if op == "host":
        s["uvw"] = np.ascontiguousarray(s["uvw"].T)
        s.update({k: torch.from_numpy(s[k]).cuda() for k in ("vis", "weights", "uvw")})
    image, beam, _ = _exact_image(case, s)
    out = dict(image=image)
    if case["beam"]:
        out["beam"] = beam
    if op == "snapshot":
        out.update(_exact_find(case, image))
    return out
