"""Bricking kernels at the edges of their walks: slots whose edge is and is
not a multiple of a block, levels smaller than a brick, rows shorter than a
run, the smallest and a large brick; cells on both sides of the 32-voxel
limit of the one-pass kernel.  Stored bricks and ranges against the oracle,
bit for bit; cells through the samples they skip."""
import numpy as np
import pytest

from conftest import gpu_renderer
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bits", [8, 16])
@pytest.mark.parametrize("dims,brick,apron", [((1, 1, 1), 8, 1), ((3, 70, 9), 8, 2), ((65, 33, 17), 16, 1),
                                              ((40, 90, 50), 37, 3), ((300, 20, 10), 256, 2), ((64, 64, 64), 32, 8)])
def test_bricks_and_ranges(dims, brick, apron, bits):
    print(f"case bricks {dims} brick {brick} apron {apron} u{bits}", flush=True)
    nx, ny, nz = dims
    rng = np.random.default_rng(nx + brick)
    v = rng.integers(1, 1 << bits, (nz, ny, nx)).astype(np.uint8 if bits == 8 else np.uint16)
    r = gpu_renderer(width=16, height=16)
    r.setVolume(v, brick, apron, 2)
    levels = O.lod_pyramid(v, 2)
    for lod, lv in enumerate(levels):
        g, _, _ = r.getDataset().getBrickLayout(lod)
        mn, mx = r.brickMinMax(lod)
        for bz in range(g[2]):
            for by in range(g[1]):
                for bx in range(g[0]):
                    ref = O.extract_brick(lv, brick, apron, bx, by, bz)
                    assert np.array_equal(r.readBrick(lod, bx, by, bz), ref), (lod, bx, by, bz)
                    assert mn[bz, by, bx] == ref.min() and mx[bz, by, bx] == ref.max(), (lod, bx, by, bz)
    r.cleanup()


@pytest.mark.parametrize("bits", [8, 16])
@pytest.mark.parametrize("brick,cell", [(32, 4), (35, 5), (32, 32), (66, 33), (60, 12), (64, 64)])
def test_cell_ranges_skip_only_air(brick, cell, bits):
    """Single voxels in air: a cell that lost one would lose it from the
    image; a cell that gained one would evaluate more samples."""
    from imagevis3d_amd import workloads
    from imagevis3d_amd.workloads import Camera
    print(f"case cells brick {brick} cell {cell} u{bits}", flush=True)
    nx, ny, nz = 131, 67, 70
    rng = np.random.default_rng(cell)
    v = np.zeros((nz, ny, nx), np.uint8 if bits == 8 else np.uint16)
    for _ in range(40):
        v[rng.integers(nz), rng.integers(ny), rng.integers(nx)] = 200
    v[0, 0, 0] = v[-1, -1, -1] = v[0, -1, 0] = v[cell, cell - 1, cell] = 200
    tf = np.zeros((256, 4), np.float32)
    tf[20:] = (0.9, 0.6, 0.3, 0.5)
    w = workloads.Workload("cells", (nx, ny, nz), bits, 0, 0, brick, 2, 1, tf, 200, 120, 1.5,
                           [Camera((0.9, 0.4, 1.2), (-0.9, -0.4, -1.2), fov=40.0)])
    r = gpu_renderer(w)
    r.setEmptySpaceCell(cell)
    r.setVolume(v, brick, 2, 1)
    r.set1DTrans(tf)
    workloads.apply(r, w, w.cameras[0])
    a, ea = r.capture(), r.frameStats().evaluated_samples
    r.setEmptySpaceSkipping(False)
    assert np.array_equal(a, r.capture()) and a.any()
    _, ns, _ = O.render(O.make_params(v, tf, **{**workloads.oracle_kwargs(w, w.cameras[0]), "brick_size": cell,
                                                "apron": 1}))
    # slack: sample positions that round to the other side of a cell face
    assert abs(int(ea) - int(ns.sum())) <= 2e-3 * ns.sum() + 64
    r.cleanup()


def test_copies_before_and_after_the_pinned_buffers():
    """A renderer's first large copies go the plain way, the later ones
    through pinned buffers in pieces: both carry every byte, odd tails
    included."""
    rng = np.random.default_rng(31)
    v = rng.integers(0, 1 << 16, (257, 259, 263)).astype(np.uint16)  # 35 MB, no multiple of a piece
    r = gpu_renderer(None, 64, 64)
    for k in range(3):
        print(f"case copy {k}", flush=True)
        r.setVolume(v + np.uint16(k), 128, 2, 1)
        assert np.array_equal(r.readLOD(0), v + np.uint16(k))
    r.cleanup()
