"""Child of test_gpu_split_room.py: malloc_limit_child.py SHIM.  One SIC whose
planes of partials do not fit the memory that is left, host- and
device-planned, host and device slabs, against the same with room."""
import ctypes as C
import os
import sys

import numpy as np

shim = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)
root = os.path.dirname(os.path.dirname(os.path.dirname(os.path.abspath(__file__))))
sys.path[:0] = [os.path.join(root, "abacus-public_amd"), os.path.join(root, "tests"), os.path.join(root, "oracle")]
import nearfield as nfm  # noqa: E402
import synth  # noqa: E402

limit, refused = C.c_size_t.in_dll(shim, "limit_bytes"), C.c_int.in_dll(shim, "refused")
cpd, ppc, x = 17, 50, 3
box = synth.uniform_box(cpd ** 3 * ppc, cpd, 3)
ell = box.mean_spacing()
n = box.slab(x).n
dev = [nfm.DeviceArray(host=box.slab(s).pos) for s in range(cpd)]
ptrs = [dev[(x - 2 + c) % cpd].ptr for c in range(5)]
# Partials of about 17^2 pencils x 5 blocks x 64 sinks x 32 B = 2.8 MiB a plane and sources of 2.1 MiB: with one
# plane 5 MiB, with five 16 MiB (each asked for with a quarter and 1 MiB on top).
for mem in (nfm.NF_MEM_DEVICE, nfm.NF_MEM_HOST):
    for planner in ("host", "device"):
        got = []
        for cap in (1 << 62, 12 << 20):
            acc = np.full((n, 4), np.nan, np.float32)
            out = nfm.DeviceArray(host=acc)
            limit.value, refused.value = 1 << 62, 0
            with nfm.NearFieldDriver(cpd, ell / 40.0, synth.fof_b2(ell), path="batched", buffers_per_device=1,
                                     max_buffer_bytes=1 << 30) as drv:
                limit.value = cap
                kw = (dict(acc_ptr=out.ptr, pos_ptrs=ptrs) if mem == nfm.NF_MEM_DEVICE
                      else dict(acc_ptr=acc.ctypes.data))
                for _ in range(2):  # (the second with the buffers of the first)
                    t = (drv.submit_slab(box, x, mem=mem, **kw) if planner == "device"
                         else drv.submit(drv.plan(box, x, mem=mem, **kw)))
                    t.wait()
                    t.release()
            limit.value = 1 << 62
            got.append(out.to_host(np.float32, (n, 4)) if mem == nfm.NF_MEM_DEVICE else acc)
            print(mem, planner, cap, "refused", refused.value, flush=True)
            assert (refused.value > 0) == (cap < 1 << 62)
        assert np.isfinite(got[0]).all()
        assert np.array_equal(got[0].view(np.uint32), got[1].view(np.uint32)), (mem, planner)
print("same without room")
