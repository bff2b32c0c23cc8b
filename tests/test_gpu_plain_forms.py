"""The plain path's short pair forms (no softening, no density term, where a
tile's bounding box rules them out) give bitwise the full form's sums.

Two particles per cell lie so far out (1e25 box lengths) that their pair terms
are exact zeros but their distance is not: at one corner and the opposite one
they stretch every tile's box over all sinks, so every tile takes the full form;
both on the +x side they leave the boxes' y and z as they are, and most tiles
take the shorter forms.  The sums must not differ."""
import numpy as np
import pytest

import nearfield as nfm
import synth
from nfhelpers import params

pytestmark = pytest.mark.gpu

FAR = np.float32(1e25)


# Partial tiles only; full and partial ones with far particles in each; and pencils of more than 64 tiles.
@pytest.mark.parametrize("per_cell", [10, 30, 900])
# (cubic Plummer is left out: its r = r2 rsqrt(r2) of an infinite r2 is not a number)
@pytest.mark.parametrize("softening", ["single_spline", "plummer", "cubic_spline"])
def test_short_forms_bitwise(softening, per_cell):
    cpd, x, R = 7, 3, 2  # slabs 1 .. 5 are the window
    rng = np.random.default_rng(per_cell)
    n = cpd * cpd * per_cell
    cells = ((rng.random((cpd, cpd * cpd, per_cell, 3)) - 0.5) / cpd).astype(np.float32)
    got = []
    for spread in (True, False):
        slabs = []
        for s in range(cpd):
            p = cells[s].copy()
            if s != x:  # the source slabs beside the sinks'
                every = min(per_cell, 58)  # a pair of them in every 64-source tile
                for a in range(every - 2, per_cell - 1, every):
                    p[:, a] = (FAR, FAR, FAR) if spread else (FAR, 0, 0)
                    p[:, a + 1] = (-FAR, -FAR, -FAR) if spread else (FAR, 0, 0)
            slabs.append(synth.Slab(p.reshape(-1, 3).T.ravel(), np.full(cpd * cpd, per_cell)))
        box = synth.Box(cpd, slabs, "far particles")
        _, b2, _ = params(box)
        dev = [nfm.DeviceArray(host=box.slab(x - R + c).pos) for c in range(2 * R + 1)]
        acc = nfm.DeviceArray(host=np.full((n, 4), np.nan, np.float32))
        with nfm.NearFieldDriver(cpd, box.mean_spacing() / 40.0, b2, softening=softening, path="plain",
                                 buffers_per_device=1, max_buffer_bytes=1 << 30) as drv:
            sic = drv.plan(box, x, pos_ptrs=[d.ptr for d in dev], acc_ptr=acc.ptr, mem=nfm.NF_MEM_DEVICE)
            drv.submit(sic, blocking=True).release()
        got.append(acc.to_host(np.float32, (n, 4)))
    assert np.isfinite(got[0]).all() and (got[0][:, 3] > 0).any()
    assert np.array_equal(got[0].view(np.uint32), got[1].view(np.uint32))
