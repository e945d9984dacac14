"""The gradient launches' LDS tables: the 2D TF's mask of texel cells with
any alpha, and small 1D TFs, at the sizes where their bits and limits can go
wrong, against the FP64 oracle; more TFs than tables, against lone views."""
import numpy as np
import pytest

from conftest import assert_parity
from imagevis3d_amd import transfer, workloads
from imagevis3d_amd.renderer import RenderMode
from oracle import oracle as O
from test_gpu_shading import LIGHT, make_renderer, medium_small, oracle_ref, render

pytestmark = pytest.mark.gpu


def sparse_tf(w, h, seed):
    """A few opaque texels, some negative alphas, colours everywhere."""
    rng = np.random.default_rng(seed)
    tf = rng.uniform(0.1, 1.0, (h, w, 4)).astype(np.float32)
    tf[..., 3] = np.where(rng.random((h, w)) < 0.08, rng.uniform(0.02, 0.2, (h, w)), 0.0)
    tf[..., 3][rng.random((h, w)) < 0.02] = -0.05
    tf[0, w - 1, 3] = tf[h - 1, 0, 3] = tf[h - 1, w - 1, 3] = 0.1  # the raster's corners
    return tf


@pytest.mark.parametrize("w,h", [(1, 1), (2, 3), (33, 1), (37, 19), (256, 256), (700, 500)])
def test_sparse_2d_tf(w, h):
    """From one texel over widths that are no multiple of a mask word to a
    mask of 43 KiB, which stays in memory."""
    print(f"case sparse 2D TF {w} x {h}", flush=True)
    wl, vol = medium_small(160, 90)
    _, mg = O.histogram_2d_exact(vol, 256, 256)
    tf2 = sparse_tf(w, h, w + h)
    r = make_renderer(wl, vol, bias_scale_tf=True, lighting=True)
    r.set2DTrans(tf2, mg)
    r.setRenderMode(RenderMode.RM_2DTRANS)
    cam = wl.cameras[4]
    img, st = render(r, wl, cam)
    scale = float(np.float32((w - 1) / float(vol.max())))
    ref8, ns, fl = oracle_ref(vol, wl, cam, None, mode=1, tf2d=tf2, max_grad=mg, tf_scale=scale,
                              lighting=True, **LIGHT)
    assert_parity(img, ref8, fl, f"sparse 2D TF {w} x {h}")
    for batch in (1, 2):  # one ray per lane
        r.setKernelTuning(batch, 4, 0)
        assert r.paint()
        assert np.array_equal(r.capture(), img)
    r.cleanup()


@pytest.mark.parametrize("n", [1, 300, 2047, 2048, 4096])
def test_lit_1d_tf_sizes(n):
    """2,047 entries and their repeated last one fill the 32 KiB of tables;
    larger TFs are read from memory."""
    print(f"case lit 1D TF of {n} entries", flush=True)
    w, vol = medium_small(160, 90)
    tf = transfer.gaussian_bumps_tf(max(n, 64), seed=5)[:n].copy()
    tf[-1] = (0.8, 0.4, 0.2, 0.05)
    r = make_renderer(w, vol, bias_scale_tf=True, lighting=True)
    r.set1DTrans(tf)
    cam = w.cameras[4]
    img, _ = render(r, w, cam)
    scale = float(np.float32((n - 1) / float(vol.max())))
    ref8, _, fl = oracle_ref(vol, w, cam, tf, tf_scale=scale, lighting=True, **LIGHT)
    assert_parity(img, ref8, fl, f"lit 1D TF {n}")
    r.cleanup()


@pytest.mark.parametrize("two_d", [False, True])
def test_more_tfs_than_tables(two_d):
    """Ten TFs in one launch: eight tables (and their 32 KiB) go to LDS, the
    others stay in memory; every view equals its own lone launch."""
    print(f"case ten TFs two_d={two_d}", flush=True)
    w, vol = medium_small(96, 54)
    _, mg = O.histogram_2d_exact(vol, 256, 256)
    r = make_renderer(w, vol, bias_scale_tf=True, lighting=True)
    if two_d:
        r.setRenderMode(RenderMode.RM_2DTRANS)
    for k in range(10):
        r.set1DTransSlot(k, transfer.gaussian_bumps_tf(200, seed=k))
        r.set2DTransSlot(k, sparse_tf(40 + k, 30, k), mg)
    views = [workloads.view_of(w.cameras[3 + k % 3], 96, 54, k) for k in range(10)]
    imgs, stats, _ = r.renderBatch(views)
    for k in range(10):
        one, st, _ = r.renderBatch([views[k]])
        assert np.array_equal(imgs[k], one[0]), k
        assert stats[k].evaluated_samples == st[0].evaluated_samples
    assert any(i.any() for i in imgs)
    r.cleanup()
