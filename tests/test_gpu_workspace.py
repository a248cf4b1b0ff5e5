"""The index build's workspaces: k-means with the least workspace it takes
against the full one (kmeans++ without and with its 8-bit copy of the keys: the
same results bit for bit), a buffer that held something else before, and the
drop-in cache giving the build's buffers back once every layer is built."""
import ctypes

import pytest
import torch

from conftest import gpu_available

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not gpu_available(), reason="needs a HIP device")]

DEV = "cuda:0"


@pytest.mark.parametrize("H,T,ks", [(8, 9001, (14, 9)), (8, 66003, (5, 6)), (8, 8200, (18,)), (8, 9003, (5, 3, 7, 4))])
def test_kmeans_with_the_least_workspace(H, T, ks):
    from adaptiveimi_amd import _lib, ops, synthetic

    print(f"[least workspace] H={H} T={T} ks={ks}", flush=True)
    keys = synthetic.make_kv(H, T, seed=T)[0].to(DEV)
    P, kmax = len(ks), max(ks)
    ref = ops.kmeans(keys, list(ks), 3, init="kmeans++")
    a = _lib.KmeansArgs(keys=keys.data_ptr(), head_stride=keys.stride(0), token_stride=keys.stride(1), kv_heads=H,
                        n_tokens=T, dim=128, parts=P, k=ops._ks(ks), max_iters=3, early_stop_min_iter=4, init_mode=2,
                        centroids=ref[0].data_ptr(), labels=ref[1].data_ptr())
    size, least = ctypes.c_size_t(), ctypes.c_size_t()
    _lib.check(_lib.lib().imi_kmeans_workspace_size(ctypes.byref(a), ctypes.byref(size)), "size")
    _lib.check(_lib.lib().imi_kmeans_min_workspace_size(ctypes.byref(a), ctypes.byref(least)), "least")
    assert least.value < size.value
    for n in (least.value, size.value - 1, size.value):
        cent = torch.zeros((H, P, kmax, 128 // P), device=DEV)
        labels = torch.empty((H, P, T), dtype=torch.int32, device=DEV)
        ws = torch.full((n,), 0xA5, dtype=torch.uint8, device=DEV)
        a.centroids, a.labels, a.workspace, a.workspace_bytes = cent.data_ptr(), labels.data_ptr(), ws.data_ptr(), n
        _lib.check(_lib.lib().imi_kmeans_execute(ctypes.byref(a), torch.cuda.current_stream().cuda_stream), "execute")
        assert torch.equal(labels, ref[1])
        assert all(torch.equal(cent[:, p, :k], ref[0][:, p, :k]) for p, k in enumerate(ks))


@pytest.mark.parametrize("side,other", [(True, False), (False, False), (False, True)])
def test_cache_gives_the_build_workspaces_back(monkeypatch, side, other):
    """Large ones, of the stream that built (the cache's own, the caller's, or
    one that the caller left before it prepares the cache); the next prefill
    makes them anew."""
    from adaptiveimi_amd import ops, synthetic
    from adaptiveimi_amd.cache_hub.adaptive_imi import adpimi_cache

    print(f"[workspaces] side={side} other={other}", flush=True)
    H, S, L = 2, 1500, 2
    layers = [[x.transpose(0, 1).unsqueeze(0).contiguous().to(DEV) for x in synthetic.make_kv(H, S, seed=i)] for i in range(L)]
    results = []
    for keep in (0, 1 << 30, 0):
        monkeypatch.setattr(ops, "_KEEP_BYTES", keep)
        cache = adpimi_cache([0], L, 1, S + 9, H, 2 * H, 128, torch.bfloat16, {str(i): DEV for i in range(L)}, 8, S, 32, 64, 4,
                             2, 0.1, 0.05, 32, 1, 1, 8, subspace_parts=2,
                             runtime_config=dict(pipeline=dict(async_build=side)))
        ops.workspace("attention", 256, torch.device(DEV))
        main = torch.cuda.current_stream()
        caller = torch.cuda.Stream() if other else main
        caller.wait_stream(main)
        with torch.cuda.stream(caller):
            for i, (k, v) in enumerate(layers):
                cache.prefill_update_kv_cache(None, k, v, i, 0)
        main.wait_stream(caller)
        stream = cache._build_stream if side else caller
        mine = {(n, stream.cuda_stream) for n in ("kmeans", "index")}
        others = {k for k in ops._WS if (k[0], k[2]) not in mine}
        assert mine <= {(n, s) for n, _, s in ops._WS}
        cache.prepare_cache()
        assert others <= set(ops._WS)
        assert len(mine & {(n, s) for n, _, s in ops._WS}) == (0 if keep == 0 else 2)
        torch.cuda.synchronize()
        results.append([x.clone() for x in cache.centroids + cache.token_perm])
    assert all(torch.equal(x, y) for r in results[1:] for x, y in zip(r, results[0]))
