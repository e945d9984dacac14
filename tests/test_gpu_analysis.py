"""Histogram, gradient and region-detail kernels at the sizes where their
walks can go wrong: rows shorter than a run of voxels, ragged ends, bins
that overflow 16-bit counters, bin counts on both sides of the LDS limits.
Every count is compared exactly with the oracle or numpy."""
import numpy as np
import pytest

from conftest import gpu_renderer
from oracle import oracle as O

pytestmark = pytest.mark.gpu

SHAPES = [(1, 1, 1), (2, 3, 4), (7, 5, 1), (8, 1, 9), (9, 16, 2), (33, 17, 9), (257, 6, 5), (70, 41, 30)]


def volume(dims, bits, seed=0):
    nx, ny, nz = dims
    rng = np.random.default_rng(seed + nx)
    v = rng.integers(0, 1 << bits, (nz, ny, nx)).astype(np.uint8 if bits == 8 else np.uint16)
    v[rng.random(v.shape) < 0.5] = 0  # air: one bin holds half the voxels
    return v


def renderer(v, brick=32, n_lod=1):
    r = gpu_renderer(width=16, height=16)
    r.setVolume(v, brick, 2, n_lod)
    return r


@pytest.mark.parametrize("bits", [8, 16])
@pytest.mark.parametrize("dims", SHAPES)
def test_histograms_small_and_ragged(dims, bits):
    print(f"case histograms {dims} u{bits}", flush=True)
    v = volume(dims, bits)
    r = renderer(v)
    assert np.array_equal(r.histogram1D(), O.histogram_1d(v))
    for nv, ng in ((256, 256), (16, 7), (2, 2)):
        h, mg = r.histogram2D(nv, ng)
        ref, ref_mg = O.histogram_2d_exact(v, nv, ng)
        assert np.array_equal(h, ref), (nv, ng)
        assert abs(mg - ref_mg) <= 1e-6 * max(ref_mg, 1e-30)
    r.cleanup()


@pytest.mark.parametrize("nv,ng", [(64, 1024), (16, 4096), (512, 256)])
def test_histogram_2d_bin_limits(nv, ng):
    """The most bins with thresholds in LDS, more gradient bins than
    thresholds, and more bins than LDS holds."""
    print(f"case 2D histogram {nv} x {ng}", flush=True)
    v = volume((70, 41, 30), 16, 3)
    r = renderer(v)
    h, _ = r.histogram2D(nv, ng)
    ref, _ = O.histogram_2d_exact(v, nv, ng)
    assert np.array_equal(h, ref)
    r.cleanup()


@pytest.mark.parametrize("bits", [8, 16])
def test_histograms_of_one_value_overflow_16_bit_counters(bits):
    """256^3 voxels nearly all alike: a work-group counts 65,536 of them in
    one bin, past what its 16-bit counter holds."""
    print(f"case one-value histograms u{bits}", flush=True)
    v = np.full((256, 256, 256), 77, np.uint8 if bits == 8 else np.uint16)
    v[100, 100, 100:110] = 200
    r = renderer(v, 256)
    assert np.array_equal(r.histogram1D(), np.bincount(v.ravel(), minlength=1 << bits))
    h, _ = r.histogram2D(256, 256)
    assert int(h.sum()) == v.size
    # gradients differ from 0 next to the ten odd voxels only
    assert np.array_equal(h, O.histogram_2d_exact(v, 256, 256)[0])
    b = r.brickHistograms(0, 16)
    assert np.array_equal(b[0], np.bincount((v >> (bits - 4)).ravel(), minlength=16))
    r.cleanup()


@pytest.mark.parametrize("bits", [8, 16])
@pytest.mark.parametrize("dims,brick,n_lod", [((33, 17, 9), 8, 3), ((70, 41, 30), 20, 3), ((65, 64, 63), 32, 2),
                                              ((21, 90, 14), 16, 4)])
def test_brick_histograms_and_region_detail(dims, brick, n_lod, bits):
    """Bricks whose edge is and is not a multiple of the run length, clipped
    bricks, several levels."""
    print(f"case bricks {dims} brick {brick} u{bits}", flush=True)
    v = volume(dims, bits, 5)
    r = renderer(v, brick, n_lod)
    levels = O.lod_pyramid(v, n_lod)
    g = [-(-n // brick) for n in dims]
    for bins in (2, 16, 64):
        hist = r.brickHistograms(0, bins)
        shift = bits - bins.bit_length() + 1
        for i in range(g[0] * g[1] * g[2]):
            x, y, z = i % g[0] * brick, i // g[0] % g[1] * brick, i // (g[0] * g[1]) * brick
            part = v[z:z + brick, y:y + brick, x:x + brick]
            assert np.array_equal(hist[i], np.bincount((part >> shift).ravel(), minlength=bins)), (i, bins)
    detail = r.regionDetail()
    zz, yy, xx = np.indices(v.shape)
    for l in range(n_lod):
        diff = np.abs(v.astype(np.int64) - levels[l][zz >> l, yy >> l, xx >> l].astype(np.int64))
        for i in range(g[0] * g[1] * g[2]):
            x, y, z = i % g[0] * brick, i // g[0] % g[1] * brick, i // (g[0] * g[1]) * brick
            mean = diff[z:z + brick, y:y + brick, x:x + brick].mean()
            # an exact sum, one rounding to FP32
            assert abs(float(detail[i, l]) - mean) <= 2.0 ** -23 * mean, (i, l)
    r.cleanup()
