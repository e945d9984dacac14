"""Samples per gather batch of the 1D march: every value a caller may set is
the one that runs, none changes the image."""
import numpy as np
import pytest

from conftest import gpu_renderer
from imagevis3d_amd import transfer, workloads
from imagevis3d_amd.renderer import Interpolant
from imagevis3d_amd.workloads import Camera

pytestmark = pytest.mark.gpu

CAM = Camera((0.9, 0.4, 1.2), (-0.9, -0.4, -1.2), fov=45.0)


def renderer(entries, w=141, h=83):
    rng = np.random.default_rng(11)
    v = rng.integers(0, 4096, (37, 70, 45)).astype(np.uint16)
    r = gpu_renderer(None, w, h)
    r.setVolume(v, 32, 2, 1)
    r.set1DTrans(transfer.gaussian_bumps_tf(entries, seed=4))
    return r


@pytest.mark.parametrize("entries", [4096, 5000])  # in LDS, and from memory
@pytest.mark.parametrize("interp", [Interpolant.Linear, Interpolant.NearestNeighbor])
def test_image_does_not_depend_on_it(interp, entries):
    print(f"case gather batches interp {interp}, {entries} TF entries", flush=True)
    r = renderer(entries)
    r.setInterpolant(interp)
    views = [workloads.view_of(CAM, 141, 83, 0)]
    ref, st, _ = r.renderBatch(views)
    assert ref[0].any()
    for batch in (1, 2, 4, 8):
        r.setKernelTuning(batch, 4, 0)
        img, s, _ = r.renderBatch(views)
        assert np.array_equal(img[0], ref[0]), batch
        assert s[0].evaluated_samples == st[0].evaluated_samples, batch
    r.cleanup()


def test_the_batch_set_is_the_one_that_runs():
    """As the autotuner reports it: the default by sampling, and what the
    caller set, 8 with trilinear sampling too."""
    print("case reported gather batches", flush=True)
    r = renderer(4096)
    views = [workloads.view_of(CAM, 141, 83, 0)]
    assert r.autotune(views, flags=0).samples_per_batch == 4
    r.setInterpolant(Interpolant.NearestNeighbor)
    assert r.autotune(views, flags=0).samples_per_batch == 8
    r.setInterpolant(Interpolant.Linear)
    for batch in (2, 4, 8):
        r.setKernelTuning(batch, 4, 0)
        assert r.autotune(views, flags=0).samples_per_batch == batch
    r.cleanup()
