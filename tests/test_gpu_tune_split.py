"""The autotuner keeps launches that split their tiles over the source pencils
apart from those that do not, and lists made on the device from the host's."""
import numpy as np
import pytest

import nearfield as nfm
from nfhelpers import params, small_uniform

pytestmark = pytest.mark.gpu


def test_split_launches_are_tuned_apart():
    cpd, x = 9, 4
    box = small_uniform(cpd=cpd, ppc=20)
    _, b2, _ = params(box)
    n = box.slab(x).n
    dev = [nfm.DeviceArray(host=box.slab(x - 2 + c).pos) for c in range(5)]
    acc = nfm.DeviceArray(host=np.full((n, 4), np.nan, np.float32))
    kw = dict(acc_ptr=acc.ptr, pos_ptrs=[d.ptr for d in dev], mem=nfm.NF_MEM_DEVICE)
    got = []
    with nfm.NearFieldDriver(cpd, box.mean_spacing() / 40.0, b2, path="batched", buffers_per_device=1,
                             max_buffer_bytes=1 << 30, max_group=1) as drv:
        for how, total in (("host", None), ("device", None), ("host", 8 << 30), ("host", None), ("device", None)):
            if how == "device":
                drv.submit_slab(box, x, blocking=True, **kw).release()
            else:
                sic = drv.plan(box, x, **kw)
                if total:
                    sic.desc.DirectTotal = total  # above the bound: nothing is split
                drv.submit(sic, blocking=True).release()
            got.append(acc.to_host(np.float32, (n, 4)).view(np.uint32))
        table = drv.autotune_table()
    assert all(np.array_equal(g, got[0]) for g in got)
    uses = {(e["split"], e["size_class"]): e["uses"] for e in table}
    assert uses == {("host", 0): 2, ("device", 0): 2, ("whole", 2): 1}, table
    assert all(e["occupancy_quarters"] == [0, 4, 0, 0] for e in table)
