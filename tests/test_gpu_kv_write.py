"""dspark_kv_write over ranges that start and end anywhere in a page: every pool byte against the documented page layout
(rows inside the range bit for bit, everything else as it was)."""
import numpy as np
import pytest

from conftest import load_host

pytestmark = pytest.mark.gpu

RANGES = [(0, 1), (0, 32), (31, 1), (31, 2), (5, 3), (8, 8), (7, 9), (1, 62), (40, 100), (33, 31), (3, 517), (64, 256)]


@pytest.mark.parametrize("KVH,D", [(8, 64), (1, 64), (4, 128), (3, 128)])
@pytest.mark.parametrize("table", ["none", "shuffled", "hole"])
def test_ranges(KVH, D, table):
    import torch
    host = load_host()
    rng = np.random.default_rng(KVH * D)
    n_pages, index = 20, host.k_page_index(D)
    for pos0, n in RANGES:
        print(f"case KVH={KVH} D={D} table={table} pos0={pos0} n={n}", flush=True)
        rows = rng.integers(0, 1 << 15, (n, 3, KVH * D)).astype(np.uint16)  # any bit patterns
        kp0 = rng.integers(0, 1 << 16, (n_pages, KVH, 32 * D)).astype(np.uint16)
        vp0 = rng.integers(0, 1 << 16, (n_pages, KVH, D, 32)).astype(np.uint16)
        bt = None if table == "none" else rng.permutation(n_pages).astype(np.int32)
        if table == "hole":
            bt[pos0 // 32] = n_pages if n % 2 else -1  # outside the pools: that page's rows are not written
        dev = lambda x: torch.from_numpy(x.view(np.int16)).cuda().view(torch.float16)  # noqa: E731
        r, kp, vp = dev(rows).view(n, -1), dev(kp0).view(n_pages, KVH, 32, D), dev(vp0)
        k, v = r[:, KVH * D:2 * KVH * D], r[:, 2 * KVH * D:]
        host.kv_write(k, v, kp, vp, pos0, None if bt is None else torch.from_numpy(bt).cuda())
        torch.cuda.synchronize()
        for t in range(n):
            lp, slot = divmod(pos0 + t, 32)
            pg = lp if bt is None else bt[lp]
            if 0 <= pg < n_pages:
                kp0[pg][:, index[slot]] = rows[t, 1].reshape(KVH, D)
                vp0[pg][:, :, slot] = rows[t, 2].reshape(KVH, D)
        assert np.array_equal(kp.view(torch.int16).cpu().numpy().view(np.uint16).reshape(kp0.shape), kp0)
        assert np.array_equal(vp.view(torch.int16).cpu().numpy().view(np.uint16), vp0)
