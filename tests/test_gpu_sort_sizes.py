"""The sort at the sizes where its route changes: one workgroup, several that count everything for themselves, three launches."""
import numpy as np
import pytest
import torch

from oracle import sorting
from pyhip_amd import moe_sorting

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,k,E,Bm,offset,masked", [
    (2049, 1, 8, 16, 0, False),            # one pair more than the single workgroup takes; a last group of one
    (683, 3, 12, 32, 1, True),             # pairs no multiple of four, ids that start 4 bytes into 16
    (1024, 8, 605, 64, 0, False),          # most experts that the counters have LDS for
    (1024, 8, 605, 64, 2, True),
    (1024, 8, 606, 64, 0, True),           # three launches for one expert more
    (16384, 8, 64, 160, 0, True),          # most pairs of the one launch: every workgroup's chunk is full
    (16384, 8, 64, 160, 3, False),
    (131073, 1, 16, 288, 0, False),        # three launches for one pair more
])
def test_sort_sizes(T, k, E, Bm, offset, masked):
    rng = np.random.default_rng(T + E)
    p = 1.0 / np.arange(1, E + 1) ** 1.1
    keys = np.log(p) + rng.gumbel(size=(T, E))
    ids = np.argpartition(-keys, k - 1, axis=1)[:, :k].astype(np.int32) if k < E else np.tile(np.arange(E, dtype=np.int32), (T, 1))
    ids[rng.random((T, k)) < 0.02] = -1                           # pairs that a caller drops by their id
    ids[rng.random((T, k)) < 0.01] = E
    w = rng.random((T, k), dtype=np.float32)
    mask = (rng.random(E) < 0.6).astype(np.int32) if masked else None
    for nloc in (None, T - 5):
        print(f"sort sizes T={T} k={k} E={E} Bm={Bm} offset={offset} masked={masked} nloc={nloc}", flush=True)
        buf = torch.empty(T * k + offset, dtype=torch.int32, device="cuda")
        t_ids = buf[offset:].view(T, k)
        t_ids.copy_(torch.from_numpy(ids))
        so, sw, se, nv, _, sched = moe_sorting(t_ids, torch.from_numpy(w).cuda(), E, 64, torch.bfloat16, Bm,
                                               None if mask is None else torch.from_numpy(mask).cuda(),
                                               None if nloc is None else torch.tensor([nloc], dtype=torch.int32, device="cuda"),
                                               alloc_moe_out=False, return_schedule=True)
        torch.cuda.synchronize()
        kept = np.where((ids >= 0) & (ids < E), ids, 0)
        on = (ids >= 0) & (ids < E) & (True if mask is None else mask[kept] != 0)
        on[T if nloc is None else nloc:] = False
        # the oracle takes ids of experts only: what is dropped goes to an expert of its own that is masked
        ids_ref = np.where(on, ids, E).astype(np.int32)
        mask_ref = np.concatenate([np.ones(E, np.int32) if mask is None else mask, [0]]).astype(np.int32)
        r_so, r_sw, r_se, r_nv = sorting.moe_sorting_ref(ids_ref, w, E + 1, Bm, expert_mask=mask_ref, num_local_tokens=nloc)
        n = so.numel()
        assert (nv.cpu().numpy().view(np.uint32) == r_nv).all()
        assert (so.cpu().numpy().view(np.uint32) == r_so[:n]).all() and (sw.cpu().numpy() == r_sw[:n]).all()
        assert (se.cpu().numpy().view(np.uint32) == r_se[:se.numel()]).all()
        blocks = (np.bincount(ids[on], minlength=E) + Bm - 1) // Bm
        assert (sched.cpu().numpy().view(np.uint32)[:E + 1] == np.concatenate([[0], np.cumsum(blocks)])).all()
