"""Several SICs in one launch that splits its tiles over the source pencils (each
with planes of its own): bitwise the accelerations of the SICs one by one, whole."""
import numpy as np
import pytest

import nearfield as nfm
import synth
from nfhelpers import params

pytestmark = pytest.mark.gpu

# (slab, rows): whole slabs, ragged row ranges, a single row.
SICS = [(2, 0, 11), (5, 0, 4), (5, 4, 11), (7, 5, 6), (2, 9, 11), (0, 0, 11), (10, 1, 8)]


def _box(cpd, radius):
    """Cells of 0 to 40 particles: pencils of tails alone, of tiles with and without one, and empty ones."""
    rng = np.random.default_rng(radius)
    slabs = []
    for _ in range(cpd):
        cnt = rng.choice([0, 0, 3, 9, 13, 40], cpd * cpd)
        local = (rng.random((int(cnt.sum()), 3)) - 0.5).astype(np.float32) / np.float32(cpd)
        slabs.append(synth.Slab(local.T.ravel(), cnt))
    return synth.Box(cpd, slabs, "cells of 0 to 40")


@pytest.mark.parametrize("planner", ["host", "device"])
@pytest.mark.parametrize("radius,sinks_per_lane,kick", [(2, 1, False), (2, 2, True), (2, 4, False), (1, 4, True),
                                                        (1, 1, False)])
def test_split_groups_bitwise(planner, radius, sinks_per_lane, kick):
    cpd, W = 11, 2 * radius + 1
    box = _box(cpd, radius)
    _, b2, _ = params(box)
    rng = np.random.default_rng(5)
    dev = [nfm.DeviceArray(host=box.slab(s).pos) for s in range(cpd)]
    far = [nfm.DeviceArray(host=rng.standard_normal((box.slab(s).n, 3)).astype(np.float32)) for s in range(cpd)]

    def run(drv, whole):
        accs = [nfm.DeviceArray(host=np.full((box.slab(x).n, 4), np.nan, np.float32)) for x, _, _ in SICS]
        tasks, sizes = [], []
        for (x, lo, hi), acc in zip(SICS, accs):
            kw = dict(pos_ptrs=[dev[(x - radius + c) % cpd].ptr for c in range(W)], acc_ptr=acc.ptr,
                      mem=nfm.NF_MEM_DEVICE)
            if kick:
                kw["kick"] = nfm.nf_kick(FarAccSlab=far[x].ptr, rescale=0.5, inv_eps3=2.0, density_rad2=float(b2))
            if planner == "device" and not whole:
                tasks.append(drv.submit_slab(box, x, lo, hi, **kw))
                continue
            sic = drv.plan(box, x, lo, hi, **kw)
            if whole:
                sic.desc.DirectTotal = 1 << 40  # above the bound: nothing is split
            tasks.append(drv.submit(sic, blocking=whole))
        for t in tasks:
            t.wait()
            sizes.append(t.stats()["group_size"])
            t.release()
        return [a.to_host(np.float32, (box.slab(x).n, 4)) for a, (x, _, _) in zip(accs, SICS)], max(sizes)

    # (waves per workgroup left to the autotuner, whose table names the kind of launch)
    setup = dict(nfradius=radius, path="batched", buffers_per_device=1, max_buffer_bytes=1 << 30,
                 sinks_per_lane=sinks_per_lane)
    with nfm.NearFieldDriver(cpd, box.mean_spacing() / 40.0, b2, **setup) as drv:
        want, _ = run(drv, True)
        assert {e["split"] for e in drv.autotune_table()} == {"whole"}
    with nfm.NearFieldDriver(cpd, box.mean_spacing() / 40.0, b2, **setup) as drv:
        got, largest = run(drv, False)
        again, _ = run(drv, False)
        assert {e["split"] for e in drv.autotune_table()} == {planner}
    assert largest > 1
    for (x, lo, hi), w, g, a in zip(SICS, want, got, again):
        first, last = box.slab(x).start[lo * cpd], box.slab(x).start[hi * cpd - 1] + box.slab(x).count[hi * cpd - 1]
        assert np.isfinite(w[first:last]).all() and np.isnan(w[:first]).all() and np.isnan(w[last:]).all()
        assert np.array_equal(g.view(np.uint32), w.view(np.uint32)), (x, lo, hi)
        assert np.array_equal(a.view(np.uint32), w.view(np.uint32)), (x, lo, hi)
