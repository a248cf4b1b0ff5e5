"""The screened E-step and the superblock member lists at the sizes where they
can go wrong: centroid counts around a 16-centroid tile, a streamed chunk and
the largest k of each width; tokens with exactly two candidates, with more (a
few per wave and whole waves), and token counts around a wave, a workgroup
and a superblock.  kmeans++ with its rows screened, the M-step's forms and the
re-seeding.  Labels, distances and centroids equal the oracle's bit for bit
(the results are defined exactly, so there is no tolerance)."""
import numpy as np
import pytest
import torch

from conftest import gpu_available

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not gpu_available(), reason="needs a HIP device")]

DEV = "cuda:0"


def _bits(t):
    return t.detach().cpu().contiguous().view(torch.int16).numpy().view(np.uint16)


def _copies(rng, cent, form):
    """Exact ties: each of a few centroids repeated once (two candidates), or
    three times more (every centroid is searched, for a few tokens or, with
    every centroid equal, for whole waves), or all of them in groups of four."""
    k = cent.shape[0]
    if form == "equal":
        cent[:] = cent[0]
    elif form == "fours":   # every token has four candidates, in queued pairs
        cent[:] = cent[np.arange(k) // 4 * 4]
        cent[2::4] *= np.float32(1 + 2.0 ** -23)
    elif form != "distinct" and k >= 8:
        n = 1 if form == "pairs" else 3
        at = rng.permutation(k)
        for i in range(0, k // (n + 1) * (n + 1), (n + 1) * (1 if form == "pairs" else 8)):
            cent[at[i + 1:i + 1 + n]] = cent[at[i]]
    return cent


@pytest.mark.parametrize("T,k,parts,form", [
    (1, 1, 2, "distinct"), (63, 2, 2, "equal"), (257, 3, 4, "distinct"), (65, 15, 4, "pairs"), (300, 16, 2, "few"),
    (511, 17, 2, "pairs"), (1000, 64, 4, "few"), (513, 65, 2, "equal"), (777, 129, 2, "pairs"), (1025, 181, 2, "few"),
    (600, 208, 2, "distinct"), (600, 209, 2, "pairs"), (900, 257, 2, "few"), (700, 511, 2, "equal"),
    (700, 512, 2, "pairs"), (65, 1, 1, "distinct"), (130, 5, 1, "equal"), (257, 63, 1, "pairs"), (600, 64, 1, "few"),
    (600, 65, 1, "distinct"), (500, 1018, 1, "pairs"), (300, 4095, 1, "few"), (257, 4096, 1, "equal"),
    (77, 16, 2, "fours"), (600, 62, 4, "fours"), (1000, 64, 2, "fours"), (513, 181, 2, "fours"), (515, 300, 4, "fours"),
    (700, 512, 2, "fours"), (400, 100, 1, "fours")])
def test_estep_edges(oracle, T, k, parts, form):
    from adaptiveimi_amd import ops, synthetic

    print(f"[estep] T={T} k={k} parts={parts} {form}", flush=True)
    H, Dp = 2, 128 // parts
    keys, _ = synthetic.make_kv(H, T, seed=T + k)
    rng = np.random.default_rng(T * 4099 + k)
    kf = oracle.bf16_to_f32(_bits(keys))
    cent = rng.standard_normal((H, parts, k, Dp)).astype(np.float32)
    for h in range(H):
        for p in range(parts):   # centroids near the keys, so that the screen has close calls
            sub = kf[h][:, p * Dp:(p + 1) * Dp]
            cent[h, p] = sub[rng.integers(0, T, k)] + 0.1 * cent[h, p]
            _copies(rng, cent[h, p], form)
    kd, cd = keys.to(DEV), torch.from_numpy(cent).to(DEV)
    plain, _ = ops.kmeans_assign(kd, cd, [k] * parts, with_distance=False)
    labels, mind = ops.kmeans_assign(kd, cd, [k] * parts)
    for h in range(H):
        for p in range(parts):
            ref, rmind, _ = oracle.estep(np.ascontiguousarray(kf[h][:, p * Dp:(p + 1) * Dp]), cent[h, p])
            assert np.array_equal(plain[h, p].cpu().numpy(), ref), (h, p)
            assert np.array_equal(labels[h, p].cpu().numpy(), ref), (h, p)
            assert np.array_equal(mind[h, p].cpu().numpy(), rmind), (h, p)


@pytest.mark.parametrize("H,T,k", [(16, 9001, 130), (16, 8449, 64), (4, 66000, 33)])
def test_estep_ivf_several_blocks_per_workgroup(oracle, H, T, k):
    """128 dims over more token blocks than the device holds at once: each
    workgroup streams the centroids again for its next block (the last one
    ragged, with waves past the last token that keep to the barriers)."""
    from adaptiveimi_amd import ops, synthetic

    print(f"[ivf blocks] H={H} T={T} k={k}", flush=True)
    assert -(-T // 256) * H > 512   # two workgroups on each of 256 CUs
    keys, _ = synthetic.make_kv(H, T, seed=T + k)
    kf = oracle.bf16_to_f32(_bits(keys))
    rng = np.random.default_rng(T + k)
    cent = np.stack([kf[h][rng.integers(0, T, (k, 3))].mean(1) for h in range(H)])[:, None].astype(np.float32)
    cent[:, :, 7 % k] = cent[:, :, 2]
    kd, cd = keys.to(DEV), torch.from_numpy(cent).to(DEV)
    plain, _ = ops.kmeans_assign(kd, cd, [k], with_distance=False)
    labels, mind = ops.kmeans_assign(kd, cd, [k])
    for h in range(H):
        ref, rmind, _ = oracle.estep(kf[h], cent[h, 0])
        assert np.array_equal(plain[h, 0].cpu().numpy(), ref), h
        assert np.array_equal(labels[h, 0].cpu().numpy(), ref), h
        assert np.array_equal(mind[h, 0].cpu().numpy(), rmind), h


@pytest.mark.parametrize("form", ["means 10", "means 100", "channels 30", "channels 300", "ball", "lengths", "huge rows"])
@pytest.mark.parametrize("T,k,parts", [(1030, 64, 2), (700, 181, 2), (515, 512, 2), (1000, 32, 4), (600, 250, 4),
                                       (600, 130, 1)])
def test_estep_undecided_tokens(oracle, T, k, parts, form):
    """Keys on which many tokens of a wave are undecided after the screen:
    offsets far above the spread, keys crowded around one, row lengths over
    three decades and rows past the magnitude bound among ordinary ones.  The
    centroids are keys and means of four, the first one (the screen's origin)
    an ordinary or a far one."""
    from adaptiveimi_amd import ops

    print(f"[undecided] T={T} k={k} parts={parts} {form}", flush=True)
    H, Dp = 2, 128 // parts
    g = torch.Generator().manual_seed(T + k)
    x = torch.randn((H, T, 128), generator=g)
    size = float(form.split()[1]) if form[-1].isdigit() else 0.0
    if form.startswith("means"):
        x = x + size * torch.randn((H, 1, 128), generator=g)
    elif form.startswith("channels"):
        x[:, :, ::16] += size
    elif form == "ball":
        x = torch.where(torch.rand((1, T, 1), generator=g) < 0.6, x[:, :1] + 0.05 * x, x)
    elif form == "lengths":
        x = x * torch.exp(2.0 * torch.randn((H, T, 1), generator=g))
    else:
        x[:, torch.rand(T, generator=g) < 0.3] *= 2.0 ** 61
    keys = x.to(torch.bfloat16)
    kf = oracle.bf16_to_f32(_bits(keys))
    rng = np.random.default_rng(T * 31 + k)
    cent = np.empty((H, parts, k, Dp), np.float32)
    for h in range(H):
        for p in range(parts):
            sub = kf[h][:, p * Dp:(p + 1) * Dp]
            cent[h, p] = sub[rng.integers(0, T, k)]
            cent[h, p, ::2] = sub[rng.integers(0, T, (cent[h, p, ::2].shape[0], 4))].mean(1)
    cent[1, :, 0] += np.float32(50.0)
    kd, cd = keys.to(DEV), torch.from_numpy(cent).to(DEV)
    plain, _ = ops.kmeans_assign(kd, cd, [k] * parts, with_distance=False)
    labels, mind = ops.kmeans_assign(kd, cd, [k] * parts)
    for h in range(H):
        for p in range(parts):
            ref, rmind, _ = oracle.estep(np.ascontiguousarray(kf[h][:, p * Dp:(p + 1) * Dp]), cent[h, p])
            assert np.array_equal(plain[h, p].cpu().numpy(), ref), (h, p)
            assert np.array_equal(labels[h, p].cpu().numpy(), ref), (h, p)
            assert np.array_equal(mind[h, p].cpu().numpy(), rmind), (h, p)


@pytest.mark.parametrize("H,T,ks,stop", [
    (1, 63, (3, 5), False), (1, 1023, (16, 7), False), (2, 1025, (33, 64), True), (2, 2049, (129, 40), False),
    (1, 4097, (8, 8, 5, 3), True), (8, 36000, (64, 64), False), (8, 70001, (45, 20), True), (1, 2050, (300,), False),
    (2, 1030, (700,), True), (1, 530000, (4, 3), False), (2, 16384, (32, 5), True), (2, 16385, (32, 5), True),
    (2, 4096, (128, 60), False), (2, 4097, (128, 60), False), (1, 300, (200, 256), True), (2, 8000, (125,), True),
    (2, 8001, (125,), False), (1, 40001, (300,), False), (1, 40001, (640,), True)])
def test_lloyd_over_superblock_edges(oracle, H, T, ks, stop):
    """Two Lloyd iterations (labels, member order and sums) around the
    superblocks' sizes (one of 1024 tokens, several, 8192 tokens each, more of
    them than the 32 the short member search covers), and around the largest
    segment whose M-step scans the labels itself and the largest mean cluster
    that one wave sums."""
    from adaptiveimi_amd import ops, synthetic

    print(f"[lloyd] H={H} T={T} ks={ks} stop={stop}", flush=True)
    keys, _ = synthetic.make_kv(H, T, seed=T)
    kw = dict(early_stop_min_iter=1, tol=0.0, early_stop_rel_tol=0.0) if stop else {}
    cent, labels, iters = ops.kmeans(keys.to(DEV), list(ks), 2, **kw)
    kf = oracle.bf16_to_f32(_bits(keys))
    for h in ([0, H - 1] if H > 1 else [0]):
        labs, cents, its = oracle.kmeans_head(kf[h], list(ks), 2, **kw)
        for p, k in enumerate(ks):
            assert int(iters[h, p]) == its[p], (h, p)
            assert np.array_equal(labels[h, p].cpu().numpy(), labs[p]), (h, p)
            assert np.array_equal(cent[h, p, :k].cpu().numpy(), cents[p]), (h, p)


@pytest.mark.parametrize("H,T,k,sizes", [
    (2, 3000, 64, (512, 513, 1100)), (1, 2500, 40, (511, 512, 1400)), (1, 9000, 290, (514, 513, 515, 516, 1023, 1025, 2500)),
    (2, 9000, 600, (513, 4097)), (1, 40001, 700, (513, 600, 20000, 512)), (1, 16000, 250, (15700,))])
def test_large_clusters_among_small(oracle, H, T, k, sizes):
    """IVF clusters around the size that one wave sums, far larger ones, several
    per segment, with fewer and more re-seeded clusters than the draws of one
    launch, and more than 32 superblocks: copies of the first rows, so that
    the sizes are what they are set to."""
    from adaptiveimi_amd import ops

    print(f"[large clusters] H={H} T={T} k={k} sizes={sizes}", flush=True)
    rng = np.random.default_rng(T + k)
    at = np.empty((H, T), np.int64)
    for h in range(H):
        own = rng.permutation(k)[:len(sizes)]
        rest = np.concatenate([np.full(n - 1, c) for n, c in zip(sizes, own)])
        small = np.setdiff1d(np.arange(k), own)
        # half of the others stay alone
        small = np.concatenate([rest, rng.choice(small[:max(1, len(small) // 2)], T - k - len(rest))])
        at[h] = np.concatenate([np.arange(k), rng.permutation(small)])
    rows = torch.randn((H, k, 128), generator=torch.Generator().manual_seed(k)).to(torch.bfloat16)
    if k > 256:   # two thirds of the rows equal: more than 256 empty clusters at k = 600 and 700
        rows[:, k // 3:] = rows[:, :1]
    keys = torch.gather(rows, 1, torch.from_numpy(at)[..., None].expand(-1, -1, 128))
    cent, labels, _ = ops.kmeans(keys.to(DEV), [k], 2)
    kf = oracle.bf16_to_f32(_bits(keys))
    for h in range(H):
        labs, cents, _ = oracle.kmeans_head(kf[h], [k], 2)
        assert np.array_equal(labels[h, 0].cpu().numpy(), labs[0]), h
        assert np.array_equal(cent[h, 0, :k].cpu().numpy(), cents[0]), h


@pytest.mark.parametrize("H,T,k", [(1, 1500, 296), (2, 1500, 297), (1, 2000, 1064), (1, 2000, 1065), (2, 2000, 1900)])
def test_reseed_slices(oracle, H, T, k):
    """40 distinct rows leave k - 40 clusters empty: around the 256 draws of the
    M-step's launch, the 768 of each later one, and more than two of those."""
    from adaptiveimi_amd import ops, synthetic

    print(f"[reseed] H={H} T={T} k={k}", flush=True)
    keys, _ = synthetic.make_kv(H, T, seed=k)
    keys = _awkward(keys, "duplicates")
    cent, labels, _ = ops.kmeans(keys.to(DEV), [k], 2)
    kf = oracle.bf16_to_f32(_bits(keys))
    for h in range(H):
        labs, cents, _ = oracle.kmeans_head(kf[h], [k], 2)
        assert np.array_equal(labels[h, 0].cpu().numpy(), labs[0]), h
        assert np.array_equal(cent[h, 0, :k].cpu().numpy(), cents[0]), h


def _awkward(keys, form):
    """Rows on which the 8-bit copy's bound is poor or degenerate."""
    k = keys.float()
    if form == "outliers":      # one huge row and one huge channel
        k[:, 1234] *= 3000.0
        k[:, :, 5] *= 500.0
    elif form == "duplicates":  # 40 distinct rows: minima fall to zero
        k = k[:, torch.arange(k.shape[1]) % 40]
    elif form == "huge":
        k *= 2.0 ** 60
    elif form == "tiny":
        k *= 2.0 ** -70
    elif form == "flat":        # no dominant channels: the copy's second half is read
        k = torch.randn(k.shape, generator=torch.Generator().manual_seed(7))
    elif form == "lengths":     # distances over too many binades for exact partial sums
        k *= torch.exp(2.0 * torch.randn(k.shape[:2], generator=torch.Generator().manual_seed(9)))[..., None]
    elif form == "steps":       # the same, the largest distances in one run of rows
        k[:, :k.shape[1] // 3] *= 2.0 ** -9
        k[:, k.shape[1] // 2:k.shape[1] // 2 + 70] *= 2.0 ** 9
    elif form == "zero":        # a whole group of zero rows
        k[:, 256:1300] = 0.0
    return k.to(torch.bfloat16)


@pytest.mark.parametrize("H,T,ks,form", [
    (8, 9001, (37, 20), ""), (8, 8193, (9, 9), "outliers"), (8, 9000, (45, 45), "duplicates"), (8, 8999, (12, 5), "huge"),
    (8, 9000, (6, 6), "tiny"), (8, 10240, (8, 30), "zero"), (1, 70001, (16, 3), ""), (8, 9000, (17, 2, 30, 1), ""),
    (8, 9007, (11, 11, 11, 11), "outliers"), (8, 8300, (70,), ""), (8, 9000, (20,), "outliers"), (1, 300100, (9, 4), ""),
    # several blocks per workgroup, four groups of 256 rows each (64, 32 and 128 dims)
    (8, 131100, (5, 4), ""), (8, 131100, (4, 5), "flat"), (8, 131100, (4, 4), "outliers"),
    (8, 70001, (4, 5, 3, 4), ""), (8, 70001, (3, 4, 4, 3), "flat"), (8, 70001, (4, 3, 3, 4), "outliers"),
    (16, 60001, (5,), ""), (16, 60001, (5,), "flat"), (16, 60001, (4,), "outliers"),
    (8, 9001, (23, 40), "flat"), (8, 8300, (9, 12, 4, 17), "flat"), (8, 9003, (30,), "flat"), (1, 70001, (12, 40), "flat"),
    (2, 4100, (33, 64), ""), (2, 257, (20, 1), ""), (1, 255, (64,), "duplicates"),
    (8, 9001, (9, 12), "lengths"), (8, 9000, (11,), "steps"), (8, 8200, (5, 9, 3, 8), "lengths"), (2, 4095, (20, 9), "lengths"),
    (2, 4097, (17,), "steps"), (1, 63, (5, 4), "lengths"), (1, 65, (6, 6), "steps"), (1, 70001, (7, 5), "steps")])
def test_plusplus_screened_rows(oracle, H, T, ks, form):
    """kmeans++ picks with the rows screened over their 8-bit copy (16 MB of
    keys and more: 64, 32 and 128 dims, ragged blocks, more blocks than one
    search round, one or both halves of the copied dims, sums that only the
    sequential loops give) and below: one Lloyd iteration from the seeds equals
    the oracle's, so every pick does."""
    from adaptiveimi_amd import ops, synthetic

    print(f"[kmeans++] H={H} T={T} ks={ks} {form}", flush=True)
    keys, _ = synthetic.make_kv(H, T, seed=T)
    keys = _awkward(keys, form)
    cent, labels, _ = ops.kmeans(keys.to(DEV), list(ks), 1, init="kmeans++")
    kf = oracle.bf16_to_f32(_bits(keys))
    for h in ([0, H - 1] if H > 1 else [0]):
        labs, cents, _ = oracle.kmeans_head(kf[h], list(ks), 1, init="kmeans++")
        for p, k in enumerate(ks):
            assert np.array_equal(labels[h, p].cpu().numpy(), labs[p]), (h, p)
            assert np.array_equal(cent[h, p, :k].cpu().numpy(), cents[p]), (h, p)


@pytest.mark.parametrize("ks,seed", [((10,), 0), ((10,), 1), ((10,), 2), ((10, 10), 0), ((10, 10), 1), ((10, 10), 2)])
def test_plusplus_weights_below_the_quotient_range(oracle, ks, seed):
    """Picks of norm 2^-53 with one non-zero dim, so that the largest weight of
    a group (its scale times the pick, 8.5e-35) is below 2^-113, where 32512
    divided by it is infinite, while the rows' distances are above the 1e-30
    the bound allows for: most rows (0.875 a, 0, ..), the first pick
    (-0.875 a, 0, ..), ten groups of entries a or a / 2 with dim 0 negated in
    every other one, which the second pick of the first kind is nearer to."""
    from adaptiveimi_amd import ops

    print(f"[kmeans++ small weights] ks={ks} seed={seed}", flush=True)
    H, T, dp, a = 1, 65536, 128 // len(ks), 2.0 ** -53
    rng = np.random.default_rng(seed)
    x = np.zeros((T, 128), np.float32)
    x[:, ::dp] = 0.875 * a
    for i, g in enumerate(rng.permutation(T // 256)[:10]):
        rows = np.where(rng.random((256, 128)) < 0.5, a, a / 2)
        if i % 2:
            rows[:, ::dp] *= -1
        x[256 * g:256 * g + 256] = rows
    number = np.arange(T, dtype=np.float32)[:, None]
    for p in range(len(ks)):   # the row that the seed's first draw takes
        first = int(oracle.kmeanspp_init(number, 1, 42 + p)[0, 0])
        x[first, p * dp:(p + 1) * dp] = 0
        x[first, p * dp] = -0.875 * a
    keys = torch.from_numpy(x)[None].to(torch.bfloat16)
    cent, labels, _ = ops.kmeans(keys.to(DEV), list(ks), 1, init="kmeans++")
    labs, cents, _ = oracle.kmeans_head(x, list(ks), 1, init="kmeans++")
    for p, k in enumerate(ks):
        assert np.array_equal(labels[0, p].cpu().numpy(), labs[p]), p
        assert np.array_equal(cent[0, p, :k].cpu().numpy(), cents[p]), p
