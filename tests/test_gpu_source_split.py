"""Tiles split over their source pencils: a launch small enough to split its
tiles gives bitwise the accelerations of one too large to, in the group path
(host- and device-planned) and in nf_execute_sic_noalloc."""
import numpy as np
import pytest

import nearfield as nfm
import synth
from nfhelpers import params

pytestmark = pytest.mark.gpu


def _box(cpd, per_cell):
    """Cells of the listed occupancies (cycled over y, z, from slab to slab)."""
    rng = np.random.default_rng(cpd)
    slabs = []
    for x in range(cpd):
        cnt = np.array([per_cell[(i + 7 * x) % len(per_cell)] for i in range(cpd * cpd)])
        local = (rng.random((int(cnt.sum()), 3)) - 0.5).astype(np.float32) / np.float32(cpd)
        slabs.append(synth.Slab(local.T.ravel(), cnt))
    return synth.Box(cpd, slabs, f"cells {per_cell}")


# Pencils of no sinks, of one tail either side of the 43-sink line (a tail of 42
# or a one-wave tile of 43 sinks), of whole tiles with and without a tail, and
# of more than 64 source blocks; few enough cells that a SIC is below the split's
# bound.
@pytest.mark.parametrize("per_cell", [(0, 0, 3), (8, 8, 9, 8, 9), (9, 8, 9), (13, 12), (64,), (27, 0, 0, 0), (900, 5)])
@pytest.mark.parametrize("radius", [1, 2])
def test_split_and_whole_tiles_bitwise(per_cell, radius):
    cpd = 7
    box = _box(cpd, per_cell)
    ell = box.mean_spacing()
    eps, b2, _ = params(box)
    x, W = 3, 2 * radius + 1
    dev = [nfm.DeviceArray(host=box.slab(s).pos) for s in range(cpd)]
    n = box.slab(x).n
    got = {}
    for how in ("host", "device", "reference"):
        acc = nfm.DeviceArray(host=np.full((n, 4), np.nan, np.float32))
        ptrs = [dev[(x - radius + c) % cpd].ptr for c in range(W)]
        with nfm.NearFieldDriver(cpd, ell / 40.0, b2, nfradius=radius, path="batched", buffers_per_device=1,
                                 max_buffer_bytes=1 << 30, sinks_per_lane=2) as drv:
            sic = drv.plan(box, x, pos_ptrs=ptrs, acc_ptr=acc.ptr, mem=nfm.NF_MEM_DEVICE)
            if how == "device":
                t = drv.submit_slab(box, x, acc_ptr=acc.ptr, pos_ptrs=ptrs, mem=nfm.NF_MEM_DEVICE)
            else:
                if how == "reference":
                    sic.desc.DirectTotal = 1 << 40  # a total above the bound: nothing is split
                t = drv.submit(sic)
            t.wait()
            t.release()
        got[how] = acc.to_host(np.float32, (n, 4))
        if how == "host":
            na = nfm.DeviceArray(host=np.full((n, 4), np.nan, np.float32))
            s2 = nfm.SetInteractionCollection(box, x, 0, cpd, radius, eps, b2, "single_spline", pos_ptrs=ptrs,
                                              acc_ptr=na.ptr, mem=nfm.NF_MEM_DEVICE)
            nfm.execute_sic_noalloc(s2)
            got["noalloc"] = na.to_host(np.float32, (n, 4))
    assert np.isfinite(got["reference"]).all()
    for how in ("host", "device", "noalloc"):
        assert np.array_equal(got[how].view(np.uint32), got["reference"].view(np.uint32)), how
