"""GPU parity of the matrix-core tile sums at the edges of their forms: grids narrower
than a tile (footprints that wrap onto it twice), kernels wider than a block, the three
sources of kernel values, tiles split into chunks, and values that are not finite.
Tolerance as for the other FP64 grids: 1e-12 of the peak."""
import numpy as np
import pytest

from fastimaging_amd import capi
from tests import simdata
from tests.helpers import peak_rel_err

pytestmark = pytest.mark.gpu


def scene(N, n, s, radius, seed):
    rng = np.random.default_rng(seed)
    uv = rng.uniform(-radius, radius, size=(n, 2))
    return uv, rng.normal(size=n) + 1j * rng.normal(size=n), rng.uniform(0.1, 2.0, size=n)


@pytest.mark.parametrize("N,n,s,os_,exact,halfplane,radius", [
    (10, 300, 2, 4, False, True, 5.0),       # the whole grid inside one tile, wrapped pieces
    (10, 300, 2, 1, True, False, 5.0),
    (22, 400, 10, 8, False, False, 11.0),    # kernel almost as wide as the grid
    (22, 400, 10, 1, True, True, 11.0),
    (66, 900, 3, 8, False, False, 33.0),     # two columns and two rows past a tile
    (128, 700, 31, 8, False, True, 60.0),    # kernels wider than a tile
    (128, 200, 60, 1, True, True, 60.0),     # exact kernels, a few entries per batch
    (128, 3000, 3, 128, False, True, 60.0),  # table too large to pad
    (256, 1023, 3, 9, False, True, 8.0),     # below the first split
    (256, 40_000, 3, 9, False, True, 8.0),   # a few heavy tiles, in chunks
    (256, 40_000, 3, 1, True, True, 8.0),
    (256, 5_000, 3, 8, False, False, 127.0),
])
def test_gpu_tile_forms(gpu, orc, N, n, s, os_, exact, halfplane, radius):
    uv, vis, w = scene(N, n, s, radius, N + n + s)
    args = (capi.KERNEL_GAUSSIANSINC, float(s), s, N, uv, vis, w)
    kw = dict(kernel_exact=exact, oversampling=os_, shift_uv=True, halfplane=halfplane, generate_beam=True)
    vg, sg, total = gpu.convolve_to_grid(*args, **kw)
    ovg, osg, ototal, _ = orc.convolve_to_grid(*args, **kw)
    assert peak_rel_err(vg, ovg) < 1e-12
    assert peak_rel_err(sg, osg) < 1e-12
    assert abs(total - ototal) <= 1e-13 * ototal


@pytest.mark.parametrize("N,n,radius", [
    (128, 2_047, 8.0),    # too few to split, all in one tile
    (128, 2_048, 8.0),    # chunks of 256
    (256, 16_385, 8.0),   # one more than chunks of 256 take
    (256, 65_535, 40.0),  # almost the full chunk
    (256, 65_536, 40.0),
    (512, 3_000, 8.0),    # more tiles: full chunks
    (64, 4_000, 30.0),    # no room for slots beside the entries
])
@pytest.mark.parametrize("exact", [False, True])
def test_gpu_tile_chunks(gpu, orc, N, n, radius, exact):
    """Heavy tiles of grids of few tiles: on both sides of each line of the chunk size."""
    uv, vis, w = scene(N, n, 3, radius, N + n)
    args = (capi.KERNEL_GAUSSIANSINC, 3.0, 3, N, uv, vis, w)
    kw = dict(kernel_exact=exact, oversampling=8, shift_uv=True, halfplane=True, generate_beam=True)
    vg, sg, total = gpu.convolve_to_grid(*args, **kw)
    ovg, osg, ototal, _ = orc.convolve_to_grid(*args, **kw)
    assert peak_rel_err(vg, ovg) < 1e-12
    assert peak_rel_err(sg, osg) < 1e-12
    assert abs(total - ototal) <= 1e-13 * ototal


@pytest.mark.parametrize("exact", [False, True])
@pytest.mark.parametrize("bad", [np.nan, np.inf])
def test_gpu_tile_values_not_finite(gpu, exact, bad):
    """A visibility that is not finite reaches its own footprint only."""
    N, s = 128, 3
    uv, vis, w = scene(N, 500, s, 60.0, 7)
    uv[100] = (20.3, 30.7)
    kw = dict(kernel_exact=exact, oversampling=8, shift_uv=False, halfplane=False, generate_beam=False)
    run = lambda v, wt: gpu.convolve_to_grid(capi.KERNEL_GAUSSIANSINC, float(s), s, N, uv, v, wt, **kw)[0]  # noqa: E731
    w0 = w.copy()
    w0[100] = 0.0
    clean = run(vis, w0)
    vis[100] = complex(bad, 1.0)
    got = run(vis, w)
    foot = np.zeros((N, N), dtype=bool)
    foot[31 + 64 - s:31 + 64 + s + 1, 20 + 64 - s:20 + 64 + s + 1] = True
    assert np.allclose(got[~foot], clean[~foot], rtol=0, atol=1e-12 * np.abs(clean).max())
    assert not np.isfinite(got[foot].real).any()
    assert np.isfinite(got[foot].imag).all()


@pytest.mark.parametrize("exact", [False, True])
@pytest.mark.parametrize("value,weight", [(np.inf, 0.0), (-np.inf, -0.0), (np.nan, 0.0), (0.0, np.inf), (1.0, np.nan)])
def test_gpu_tile_products_not_finite(gpu, exact, value, weight):
    """A visibility whose product with its weight is not finite reaches its own footprint only,
    also where neither or only one of the two is finite."""
    N, s = 128, 3
    uv, vis, w = scene(N, 500, s, 60.0, 8)
    uv[100] = (20.3, 30.7)
    kw = dict(kernel_exact=exact, oversampling=8, shift_uv=False, halfplane=False, generate_beam=True)
    run = lambda v, wt: gpu.convolve_to_grid(capi.KERNEL_GAUSSIANSINC, float(s), s, N, uv, v, wt, **kw)[:2]  # noqa: E731
    w[100] = 0.0
    vis[100] = 0.0
    clean = run(vis, w)
    vis[100], w[100] = complex(0.0, value), weight
    foot = np.zeros((N, N), dtype=bool)
    foot[31 + 64 - s:31 + 64 + s + 1, 20 + 64 - s:20 + 64 + s + 1] = True
    got = run(vis, w)
    for g, c in zip(got, clean):
        assert np.allclose(g[~foot], c[~foot], rtol=0, atol=1e-12 * np.abs(c).max())
    assert not np.isfinite(got[0][foot].imag).any()
    assert np.isfinite(got[1][foot]).any() == np.isfinite(weight)


def test_gpu_split_tiles_in_batches(gpu):
    """Fused batches split heavy tiles too: the same images as single calls."""
    ctx, items, singles, bufs = gpu, [], [], []
    for k, (N, n) in enumerate(((256, 30_000), (512, 3_000), (256, 1_500))):
        snap = simdata.snapshot(N, 2.0, n, 3, seed=simdata.seed_for(0, 40 + k))
        snap["uvw"][:, :2] *= 0.05  # most visibilities in one or two tiles
        pars = capi.imager_pars(N, 2.0)
        b = [ctx.malloc(x) for x in (16 * n, 8 * n, 24 * n, 8 * N * N, 8 * N * N)]
        for p, a in zip(b, (snap["vis"], snap["weights"], np.asfortranarray(snap["uvw"]))):
            ctx.htod(p, a)
        it = capi.BatchItem()
        it.img_pars, it.n_vis = pars, n
        it.d_vis, it.d_vis_weights, it.d_uvw_lambda, it.d_image, it.d_beam = (p.value for p in b)
        items.append(it)
        bufs.append(b)
        singles.append(ctx.image_visibilities(snap["vis"], snap["weights"], snap["uvw"], pars))
    ctx.image_batch(items, flags=capi.BATCH_FUSED)
    for it, b, (image, beam) in zip(items, bufs, singles):
        N = it.img_pars.image_size
        for p, ref in ((b[3], image), (b[4], beam)):
            out = np.empty((N, N), order="F")
            ctx.dtoh(out, p)
            assert peak_rel_err(out, ref) < 1e-12
        for p in b:
            ctx.free(p)
