"""The batched pair forms either side of their pieces: isolated pairs at
separations around 1 and 2 softening lengths, inside a cell and across a cell
boundary, in one box large enough that some blocks take the unsoftened form and
some the full one, against the FP64 oracle."""
import numpy as np
import pytest

import nearfield as nfm
import pyoracle as po
import synth
from nfhelpers import R, rel_err

pytestmark = pytest.mark.gpu

U = (0.0, 0.3, 0.999, 1.001, 1.5, 1.999, 2.001, 3.0, 6.0)


def _pairs_box(softening, cpd=7):
    """(box, softening length, e): one pair per listed r/e, each in its own
    part of the box; odd pairs straddle the cell boundary in x."""
    soft = 0.004
    _, e = synth.eps_param(softening, soft)
    rng = np.random.default_rng(7)
    pos = []
    for i, u in enumerate(U):
        c = synth.cell_centre(np.array([3, (2 * i) % cpd, (3 * i + 1) % cpd]), cpd)
        if i % 2:
            c = c + np.array([0.5 / cpd - 0.4 * u * e, 0.0, 0.0])
        d = np.array([1.0, 0.0, 0.0]) if i % 2 else rng.standard_normal(3)
        pos += [c, c + u * e * d / np.linalg.norm(d)]
    return synth.box_from_global(np.array(pos), cpd), soft, e


@pytest.mark.parametrize("softening", sorted(synth.SOFTENINGS))
def test_pair_pieces_vs_fp64(softening):
    box, soft, e = _pairs_box(softening)
    eps, _ = synth.eps_param(softening, soft)
    b2 = synth.fof_b2(2.5 * e / 0.25)  # FOF radius 2.5 e
    with nfm.NearFieldDriver(box.cpd, soft, b2, softening=softening, path="batched", buffers_per_device=1,
                             max_buffer_bytes=1 << 30, sinks_per_lane=2) as drv:
        for x in (3, 4):
            n = box.slab(x).n
            acc = np.full((n, 4), np.nan, np.float32)
            drv.execute_slab(box, x, acc, blocking=True)
            drv.finalize(x)
            sl, ix, ce = po.slab_sinks(box, x)
            ref = po.direct_f64(box, R, softening, eps, b2, sl, ix, ce)
            # A separation is known to 3 roundings of coordinates, each
            # of at most 0.36 (2.5 cells), against r >= 0.3 e = 1.2e-3; g varies as up to r^-3; ten
            # more roundings in the arithmetic.  Coincident pairs (u = 0) feel only the other pairs.
            tol = 4 * 3 * 0.36 * 2.0 ** -25 / (0.3 * 0.004) + 10 * 2.0 ** -24
            assert rel_err(acc, ref).max() <= tol
            assert np.abs(acc[:, 3] - ref[:, 3]).max() <= 1e-5 * float(b2) * len(U)


@pytest.mark.parametrize("softening", sorted(synth.SOFTENINGS))
def test_plain_pair_pieces_vs_fp64(softening):
    """The same on the plain path, whose tiles leave out branches by their boxes."""
    box, soft, e = _pairs_box(softening)
    eps, _ = synth.eps_param(softening, soft)
    b2 = synth.fof_b2(2.5 * e / 0.25)
    with nfm.NearFieldDriver(box.cpd, soft, b2, softening=softening, path="plain", buffers_per_device=1,
                             max_buffer_bytes=1 << 30) as drv:
        for x in (3, 4):
            n = box.slab(x).n
            acc = np.full((n, 4), np.nan, np.float32)
            drv.execute_slab(box, x, acc, blocking=True)
            drv.finalize(x)
            sl, ix, ce = po.slab_sinks(box, x)
            ref = po.direct_f64(box, R, softening, eps, b2, sl, ix, ce)
            # as above, with the FLOAT cell offsets' rounding in each coordinate too; the cubic
            # spline's middle piece cancels to a 50th of its terms near r = 2 e
            tol = 2 * 4 * 3 * 0.36 * 2.0 ** -25 / (0.3 * 0.004) + 10 * 50 * 2.0 ** -24
            assert rel_err(acc, ref).max() <= tol
            assert np.abs(acc[:, 3] - ref[:, 3]).max() <= 1e-5 * float(b2) * len(U)


@pytest.mark.parametrize("path,s", [("plain", 0), ("batched", 1), ("batched", 2), ("batched", 4)])
def test_source_counts_vs_fp64(path, s):
    """Lone cells around the tile loop's source batches and the blocks' ends
    (16, 64), each in a pencil whose other cells are empty."""
    cpd, soft, counts = 9, 0.03, (1, 15, 16, 17, 48, 63, 64, 65, 80)
    rng = np.random.default_rng(16)
    pos = [synth.cell_centre(np.array([4, 3 * (i // 3), 3 * (i % 3)]), cpd) + (rng.random((n, 3)) - 0.5) * (0.9 / cpd)
           for i, n in enumerate(counts)]
    box = synth.box_from_global(np.concatenate(pos), cpd)
    eps, e = synth.eps_param("single_spline", soft)
    b2 = synth.fof_b2(0.1)
    with nfm.NearFieldDriver(cpd, soft, b2, softening="single_spline", path=path, buffers_per_device=1,
                             max_buffer_bytes=1 << 30, **({"sinks_per_lane": s} if s else {})) as drv:
        acc = np.full((box.slab(4).n, 4), np.nan, np.float32)
        drv.execute_slab(box, 4, acc, blocking=True)
        drv.finalize(4)
    sl, ix, ce = po.slab_sinks(box, 4)
    ref = po.direct_f64(box, R, "single_spline", eps, b2, sl, ix, ce)
    # Per source, in the output's units (e^3 a): the force's slope is at most 10, a separation
    # is off by 3 roundings of coordinates of at most 0.36, and ten more roundings of a term of
    # at most 2.5 e; the plain path's FLOAT cell offsets double the first.
    tol = max(counts) * (2 * 10 * 3 ** 0.5 * 3 * 0.36 * 2.0 ** -25 + 10 * 2.0 ** -24 * 2.5 * e)
    assert np.abs(acc[:, :3] - ref[:, :3]).max() <= tol
    assert np.abs(acc[:, 3] - ref[:, 3]).max() <= 1e-5 * float(b2) * max(counts)
