"""Record offsets and the total, formed by the forward march for small batches and by
the scan for larger ones: both equal the running sum of the counts, at ray counts
around a workgroup's rays, around the scan's chunk and on both sides of the
change, and in a second step on the same workspace."""
import ctypes as C

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_rays", [1, 3, 4, 5, 4095, 4096, 4097, 16385])
def test_offsets_are_running_sums(n_rays):
    from plenvdb_amd import lib, scenes
    from plenvdb_amd.fused import FusedTrainer

    tr = FusedTrainer(scenes.make_scene("c2", n_rays=n_rays))
    ptr = [C.c_void_p() for _ in range(7)]
    for _ in range(2):
        tr.forward_backward()
        torch.cuda.synchronize()
        lib.call("pvdb_fused_records", tr.topo.handle, C.byref(tr.desc), *[C.byref(p) for p in ptr])
        count, offset, total = (
            tr.workspace[p.value - tr.workspace.data_ptr():][:4 * k].view(torch.int32).cpu().numpy()
            for p, k in zip(ptr[4:], (n_rays, n_rays, 1)))
        print("[case]", n_rays, "rays,", total[0], "records", flush=True)
        run = np.concatenate([[0], np.cumsum(count, dtype=np.int64)])
        np.testing.assert_array_equal(offset, run[:-1])
        assert total[0] == run[-1] and (n_rays < 8 or run[-1] > 0)
