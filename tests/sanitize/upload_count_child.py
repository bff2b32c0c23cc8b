"""Child of test_gpu_noalloc_upload.py: upload_count_child.py SHIM.  Prints the
bytes nf_execute_sic_noalloc uploads for one SIC whose tiles all stay whole: as
part of a launch large enough never to split a tile, of one that might, and (as
planned) of one whose tiles are all split."""
import ctypes as C
import os
import sys

import numpy as np

shim = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)
root = os.path.dirname(os.path.dirname(os.path.dirname(os.path.abspath(__file__))))
sys.path[:0] = [os.path.join(root, "abacus-public_amd")]
import nearfield as nfm  # noqa: E402
import synth  # noqa: E402

uploaded = C.c_size_t.in_dll(shim, "uploaded")
cpd, ppc, x = 17, 50, 3
box = synth.uniform_box(cpd ** 3 * ppc, cpd, 3)
ell = box.mean_spacing()
eps, _ = synth.eps_param("single_spline", ell / 40.0)
n = box.slab(x).n
dev = [nfm.DeviceArray(host=box.slab(x - 2 + c).pos) for c in range(5)]
out = []
for total in (1 << 40, 7900000000, None):
    acc = nfm.DeviceArray(host=np.full((n, 4), np.nan, np.float32))
    sic = nfm.SetInteractionCollection(box, x, 0, cpd, 2, eps, synth.fof_b2(ell), "single_spline",
                                       pos_ptrs=[d.ptr for d in dev], acc_ptr=acc.ptr, mem=nfm.NF_MEM_DEVICE)
    if total:
        sic.desc.DirectTotal = total
    uploaded.value = 0
    nfm.execute_sic_noalloc(sic)
    a = acc.to_host(np.float32, (n, 4))
    out.append((uploaded.value, a.view(np.uint32)))
    assert np.isfinite(a).all() and np.array_equal(out[0][1], out[-1][1])
print("uploaded", *(b for b, _ in out))
