"""The superblock cell sort of the index build at its edges: token counts
around a wave, a superblock of 1024 and of 8192 tokens, past 512 superblocks
of 8192 (where the largest k leaves no room to stage the slice), k = 1, odd and largest
k per subspace (the digits of a cell id come from 32-bit divisions), the
largest IVF cluster count, one cell holding everything and labels in runs.
Order, counts and offsets equal the stable host sort exactly."""
import math

import numpy as np
import pytest
import torch

from conftest import gpu_available

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not gpu_available(), reason="needs a HIP device")]

DEV = "cuda:0"


@pytest.mark.parametrize("H,T,ks,form", [
    (1, 1, (1, 1), ""), (2, 63, (7, 3), ""), (1, 1023, (512, 512), ""), (3, 1025, (181, 181), ""), (1, 4097, (1, 9), ""),
    (2, 2049, (3, 1, 5, 7), ""), (1, 9001, (64, 64, 64, 64), ""), (8, 70003, (97, 33), ""), (8, 66000, (32, 32, 31, 5), ""),
    (2, 5000, (4096,), ""), (1, 3001, (1,), ""), (4, 9000, (128, 128), "one"), (4, 20000, (45, 64), "runs"),
    (1, 540001, (90, 90), ""), (1, 4200003, (4096,), ""), (1, 4200003, (181, 181), "")])
def test_cell_order_counts_offsets(H, T, ks, form):
    from adaptiveimi_amd import ops

    print(f"[cell sort] H={H} T={T} ks={ks} {form}", flush=True)
    rng = np.random.default_rng(T + len(ks))
    P = len(ks)
    lab = np.stack([rng.integers(0, k, (H, T)) for k in ks], 1).astype(np.int32)
    if form == "one":
        lab[:] = (np.array(ks) - 1)[None, :, None]
    elif form == "runs":
        lab = np.stack([np.broadcast_to((np.arange(T) // (50 * (p + 1))) % k, (H, T)) for p, k in enumerate(ks)], 1)
        lab = np.ascontiguousarray(lab, np.int32)
    keys = (torch.arange(H * T * 128, device=DEV) % 251).to(torch.bfloat16).view(H, T, 128)
    cent = torch.zeros((H, P, max(ks), 128 // P), device=DEV)
    idx = ops.build_index(keys, keys, cent, torch.from_numpy(lab).to(DEV), list(ks), compact=False)
    cell = np.zeros((H, T), np.int64)
    for p, k in enumerate(ks):
        cell = cell * k + lab[:, p]
    n = math.prod(ks)
    for h in range(H):
        order = np.argsort(cell[h], kind="stable")
        count = np.bincount(cell[h], minlength=n)
        assert np.array_equal(idx["perm"][h].cpu().numpy(), order), h
        assert np.array_equal(idx["cell_count"][h].cpu().numpy(), count), h
        assert np.array_equal(idx["cell_offset"][h].cpu().numpy(), np.concatenate([[0], np.cumsum(count)])), h
        assert torch.equal(idx["list_keys"][h], keys[h][idx["perm"][h].long()])
