// IMI cell index on gfx950: stable cell order, CSR over global cells, compact
// metadata and the K/V row permutation.
//
// Reference: library/AdaptiveIMI/cpp_extensions/src/reorganize_core.cpp
//   build_compact_reorg_input   18-85 (2-way), 87-176 (4-way)
//   reorganize_single_head      234-311 (stable counting sort by compact cell,
//                               then the K/V row copy)
// and the padded metadata of pipeline_bindings.cpp:206-276 /
// indexing.py:108-174.
//
// The cell order is produced by an LSD sort with one stable counting pass per
// subspace label (last subspace first), which yields tokens ordered by
// (l0, l1, ..., token) = (global cell id, token): the reference's CSR order,
// because compact ids are ranks of global ids.  The first pass reads every
// label once, in token order, and carries each token's global cell id along,
// so the later passes read sequentially too (no gathers by token).  IVF (one subspace, the
// cluster label is the cell id; build_compact_reorg_input_ivf, 178-231) is
// the one-pass case.
#include "imi_common.hpp"
#include "imi_sort.hpp"

namespace imi {
namespace {

struct IxParams {
    const int32_t* labels;  // [H][P][T]
    int H, T, P, kmax;
    int k[4];
    int64_t ncells;
    int sbt, nsb;    // tokens per superblock, superblocks per head
    int32_t* hist;   // [H][k][nsb] digit counts of a pass, then places
    int32_t* cid;    // [H][ncells] compact id scratch
    int32_t* sums;   // [H][nchunk][2] per-chunk row and occupied totals
};

constexpr int kIvfMaxK = 4096;   // IVF clusters per head

// One LSD pass: items in the order of the pass before (token and cell id;
// null in the first pass, where item i is token i), sorted by the label of
// subspace p.  The label is (cell / div) % k with exact 32-bit division:
// mulhi by ceil(2^32 / d) is the quotient or one above it for cells < 2^26.
struct IxPass {
    int p;
    const int32_t* tok;
    const int32_t* cell;
    int32_t* tok_out;
    int32_t* cell_out;
    uint32_t div, div_magic;   // product of the k after subspace p
    uint32_t k, k_magic;
    bool stage;                // the slice is staged in LDS (place_lds_bytes)
};

__device__ __forceinline__ uint32_t quot(uint32_t n, uint32_t d, uint32_t magic) {
    if (d == 1) return n;
    const uint32_t q = __umulhi(n, magic);
    return q * d > n ? q - 1 : q;
}

// The pass's digit of item i of head h.
__device__ __forceinline__ int pass_digit(const IxParams& a, const IxPass& s, int h, int64_t i) {
    if (s.cell == nullptr) return a.labels[(static_cast<int64_t>(h) * a.P + s.p) * a.T + i];
    const uint32_t q = quot(static_cast<uint32_t>(s.cell[static_cast<int64_t>(h) * a.T + i]), s.div, s.div_magic);
    return static_cast<int>(q - quot(q, s.k, s.k_magic) * s.k);
}

// A pass is three launches: digit counts of each superblock, an exclusive scan
// of them in (digit, superblock) order, and the places.  What bounds it is the
// latency of one superblock's loads and LDS rounds up to 128k tokens, and past
// that the scattered writes.  Superblocks of 1024 .. 8192 items keep the scan
// short (at 256 items per histogram, one workgroup per head scanned 2k values
// per 512 tokens) and write each digit's items in runs; carrying the cell id
// makes every read sequential.  Measured per pass against per-256 histograms
// with labels gathered by token: 8 x 128k tokens, k = 90: 4.6 + 4.1 + 16.9 us
// (was 10.2 + 14.9 + 11.4); 8 x 1M: 10 + 6.5 + 89 us (was 85 + 210 + 104); the
// scan of 8 x 512k at k = 256: 4.7 us (was 180).  All passes of a short head on
// one workgroup, one launch in place of six, took longer: 35 us against 29 at
// 8k tokens.

// Digit counts of each superblock.
__global__ __launch_bounds__(1024) void ix_hist_kernel(IxParams a, IxPass s) {
    extern __shared__ int smem_i[];
    const int h = blockIdx.y, sb = blockIdx.x, k = static_cast<int>(s.k);
    for (int c = threadIdx.x; c < k; c += blockDim.x) smem_i[c] = 0;
    __syncthreads();
    const int base = sb * a.sbt, m = min(a.sbt, a.T - base);
    for (int i0 = 0; i0 < m; i0 += 4 * blockDim.x) {
        int d[4];
#pragma unroll
        for (int u = 0; u < 4; ++u)
            d[u] = pass_digit(a, s, h, base + min(i0 + u * static_cast<int>(blockDim.x) + static_cast<int>(threadIdx.x), m - 1));
#pragma unroll
        for (int u = 0; u < 4; ++u)
            if (i0 + u * blockDim.x + threadIdx.x < m) atomicAdd(&smem_i[d[u]], 1);
    }
    __syncthreads();
    for (int c = threadIdx.x; c < k; c += blockDim.x)
        a.hist[(static_cast<int64_t>(h) * k + c) * a.nsb + sb] = smem_i[c];
}

__global__ __launch_bounds__(1024) void ix_scan_kernel(IxParams a, int k) {
    __shared__ int sh[40];
    const int h = blockIdx.x;
    block_exclusive_scan_1024(a.hist + static_cast<int64_t>(h) * k * a.nsb, static_cast<int64_t>(k) * a.nsb, sh);
}

// Places of each superblock's items: its slice in digit order, each digit's
// run at its scanned place.  Staged in LDS, so that each digit's run is written
// together, where the slice fits (always up to 4M tokens per head).
inline size_t place_lds_bytes(int waves, int k, int sbt, bool stage) {
    return (static_cast<size_t>(waves + 2) * k + 32) * sizeof(int) + (stage ? 4 * static_cast<size_t>(sbt) : 0);
}

__global__ __launch_bounds__(1024) void ix_place_kernel(IxParams a, IxPass s) {
    extern __shared__ int smem_i[];
    const int k = static_cast<int>(s.k);
    int* cnt = smem_i;                              // [waves][k]
    int* first = cnt + (blockDim.x >> 6) * k;       // [k] first place in the slice
    int* dst = first + k;                           // [k] first place in the output
    int* wsum = dst + k;                            // [16]
    uint16_t* item = reinterpret_cast<uint16_t*>(wsum + 32);   // [sbt]
    uint16_t* dig = item + a.sbt;                              // [sbt]
    const bool stage = s.stage;
    const int h = blockIdx.y, sb = blockIdx.x;
    const int base = sb * a.sbt, m = min(a.sbt, a.T - base);
    const int64_t hT = static_cast<int64_t>(h) * a.T;
    for (int c = threadIdx.x; c < k; c += blockDim.x) dst[c] = a.hist[(static_cast<int64_t>(h) * k + c) * a.nsb + sb];
    const auto write = [&](int i, int64_t to) {   // local item i
        const int64_t at = hT + base + i;
        int cell = 0;
        if (s.cell) {
            cell = s.cell[at];
        } else {
            for (int p = 0; p < a.P; ++p) cell = cell * a.k[p] + a.labels[(static_cast<int64_t>(h) * a.P + p) * a.T + base + i];
        }
        s.tok_out[hT + to] = s.tok ? s.tok[at] : base + i;
        s.cell_out[hT + to] = cell;
    };
    // (its first barrier also publishes dst)
    superblock_sort(
        m, a.sbt, k, cnt, wsum, [&](int i) { return pass_digit(a, s, h, base + i); },
        [&](int c, int f) { first[c] = f; },
        [&](int i, int at) {
            const int d = pass_digit(a, s, h, base + i);
            if (stage) {
                item[at] = static_cast<uint16_t>(i);
                dig[at] = static_cast<uint16_t>(d);
            } else {
                write(i, dst[d] + (at - first[d]));
            }
        });
    if (!stage) return;
    __syncthreads();
    for (int i = threadIdx.x; i < m; i += blockDim.x) {
        const int d = dig[i];
        write(item[i], dst[d] + (i - first[d]));
    }
}

__global__ void ix_zero_kernel(int32_t* x, int64_t n) {
    for (int64_t i = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x; i < n;
         i += static_cast<int64_t>(gridDim.x) * blockDim.x)
        x[i] = 0;
}

// Cell counts over the sorted cell ids: equal cells are contiguous, so each
// wave adds one count per run of equal cells (one atomic per run instead of
// one per token).  Reading sorted ids: 16 us at 8 x 1M tokens, 160 when each
// token's labels were gathered in cell order.
__global__ __launch_bounds__(256) void ix_count_kernel(IxParams a, const int32_t* cells, int32_t* count) {
    const int h = blockIdx.y;
    const int i = blockIdx.x * 256 + threadIdx.x;
    const int lane = lane_id();
    const int c = i < a.T ? cells[static_cast<int64_t>(h) * a.T + i] : -1;
    const int cp = __shfl(c, lane > 0 ? lane - 1 : 0);
    const uint64_t starts = __builtin_amdgcn_ballot_w64(lane == 0 || c != cp);
    if (c >= 0 && (lane == 0 || c != cp)) {
        const uint64_t after = lane < 63 ? starts >> (lane + 1) : 0ull;
        const int len = after ? __builtin_ctzll(after) + 1 : 64 - lane;
        atomicAdd(&count[static_cast<int64_t>(h) * a.ncells + c], len);
    }
}

constexpr int kOffCells = 8192;                 // cells per workgroup of the offset scan
constexpr int kOffPT = kOffCells / 256;         // 32 consecutive cells per thread

// Inclusive scan of two ints over a 256-thread block; totals in tx / ty.
__device__ __forceinline__ void block_scan2_256(int& x, int& y, int* sh, int& tx, int& ty) {
    const int ix = wave_incl_scan(x), iy = wave_incl_scan(y);
    const int w = threadIdx.x >> 6;
    if (lane_id() == 63) {
        sh[w] = ix;
        sh[4 + w] = iy;
    }
    __syncthreads();
    int bx = 0, by = 0;
    tx = 0;
    ty = 0;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        if (j < w) {
            bx += sh[j];
            by += sh[4 + j];
        }
        tx += sh[j];
        ty += sh[4 + j];
    }
    x = bx + ix;
    y = by + iy;
    __syncthreads();
}

// Per chunk of kOffCells global cells: the row count and the occupied cells.
__global__ __launch_bounds__(256) void ix_chunk_sums_kernel(IxParams a, const int32_t* count, int32_t* sums,
                                                            int nchunk) {
    __shared__ int sh[8];
    const int h = blockIdx.y, chunk = blockIdx.x, tid = threadIdx.x;
    const int32_t* c = count + static_cast<int64_t>(h) * a.ncells;
    int t = 0, o = 0;
#pragma unroll 8
    for (int u = 0; u < kOffPT; ++u) {
        const int64_t g = static_cast<int64_t>(chunk) * kOffCells + u * 256 + tid;
        const int v = g < a.ncells ? c[g] : 0;
        t += v;
        o += v > 0 ? 1 : 0;
    }
    int tt, to;
    block_scan2_256(t, o, sh, tt, to);
    if (tid == 0) {
        sums[(static_cast<int64_t>(h) * nchunk + chunk) * 2 + 0] = tt;
        sums[(static_cast<int64_t>(h) * nchunk + chunk) * 2 + 1] = to;
    }
}

// offsets[h][g] = exclusive prefix of count (offsets[h][ncells] = T); when
// compact metadata is requested also cid[h][g] = exclusive prefix of the
// occupied flags and n_active[h].  One workgroup per chunk: its base is the
// sum of the chunk totals before it, then 32 consecutive cells per thread.
__global__ __launch_bounds__(256) void ix_offsets_kernel(IxParams a, const int32_t* count, int32_t* offset,
                                                         int32_t* n_active, const int32_t* sums, int nchunk) {
    __shared__ int sh[8];
    const int h = blockIdx.y, chunk = blockIdx.x, tid = threadIdx.x;
    const int32_t* c = count + static_cast<int64_t>(h) * a.ncells;
    int32_t* o = offset + static_cast<int64_t>(h) * (a.ncells + 1);
    const int64_t g0 = static_cast<int64_t>(chunk) * kOffCells + static_cast<int64_t>(tid) * kOffPT;
    int v[kOffPT];
    if (g0 + kOffPT <= a.ncells && (reinterpret_cast<uintptr_t>(c + g0) & 15) == 0) {
#pragma unroll
        for (int u = 0; u < kOffPT / 4; ++u) {
            const int4 q = reinterpret_cast<const int4*>(c + g0)[u];
            v[4 * u + 0] = q.x;
            v[4 * u + 1] = q.y;
            v[4 * u + 2] = q.z;
            v[4 * u + 3] = q.w;
        }
    } else {
#pragma unroll
        for (int u = 0; u < kOffPT; ++u) v[u] = g0 + u < a.ncells ? c[g0 + u] : 0;
    }
    int bt = 0, bo = 0;
    for (int i = tid; i < chunk; i += 256) {
        bt += sums[(static_cast<int64_t>(h) * nchunk + i) * 2 + 0];
        bo += sums[(static_cast<int64_t>(h) * nchunk + i) * 2 + 1];
    }
    int btt, bot;
    block_scan2_256(bt, bo, sh, btt, bot);
    int lt = 0, lo = 0;
#pragma unroll
    for (int u = 0; u < kOffPT; ++u) {
        lt += v[u];
        lo += v[u] > 0 ? 1 : 0;
    }
    int et = lt, eo = lo, tt, to;
    block_scan2_256(et, eo, sh, tt, to);
    int rt = btt + et - lt, ro = bot + eo - lo;
    int32_t* id = a.cid ? a.cid + static_cast<int64_t>(h) * a.ncells : nullptr;
    int ov[kOffPT], iv[kOffPT];
#pragma unroll
    for (int u = 0; u < kOffPT; ++u) {
        ov[u] = rt;
        iv[u] = ro;
        rt += v[u];
        ro += v[u] > 0 ? 1 : 0;
    }
    // 16-byte stores where the row allows them (the offset rows start at
    // h * (ncells + 1), so their alignment varies with h)
    const bool o_vec = g0 + kOffPT <= a.ncells && (reinterpret_cast<uintptr_t>(o + g0) & 15) == 0;
    const bool i_vec = id && g0 + kOffPT <= a.ncells && (reinterpret_cast<uintptr_t>(id + g0) & 15) == 0;
#pragma unroll
    for (int u = 0; u < kOffPT / 4; ++u) {
        if (o_vec) reinterpret_cast<int4*>(o + g0)[u] = make_int4(ov[4 * u], ov[4 * u + 1], ov[4 * u + 2], ov[4 * u + 3]);
        if (i_vec) reinterpret_cast<int4*>(id + g0)[u] = make_int4(iv[4 * u], iv[4 * u + 1], iv[4 * u + 2], iv[4 * u + 3]);
    }
#pragma unroll
    for (int u = 0; u < kOffPT; ++u) {
        if (g0 + u >= a.ncells) continue;
        if (!o_vec) o[g0 + u] = ov[u];
        if (id && !i_vec) id[g0 + u] = iv[u];
    }
    if (chunk == nchunk - 1 && tid == 0) {
        o[a.ncells] = btt + tt;
        if (id) n_active[h] = bot + to;
    }
}

struct CompactOut {
    int n_c;
    const float* cent;  // [H][P][kmax][DP]
    int DP, D;
    int32_t* gid;
    int32_t* size;
    int32_t* offset;
    float* merged;
    uint8_t* mask;
};

// One thread per global cell: an occupied cell writes its compact slot.
__global__ __launch_bounds__(256) void ix_compact_fill_kernel(IxParams a, CompactOut o, const int32_t* count,
                                                              const int32_t* offset) {
    const int h = blockIdx.y;
    const int64_t g = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
    if (g >= a.ncells) return;
    const int cnt = count[static_cast<int64_t>(h) * a.ncells + g];
    if (cnt == 0) return;
    const int c = a.cid[static_cast<int64_t>(h) * a.ncells + g];
    const int64_t hc = static_cast<int64_t>(h) * o.n_c + c;
    o.gid[hc] = static_cast<int32_t>(g);
    o.size[hc] = cnt;
    o.offset[static_cast<int64_t>(h) * (o.n_c + 1) + c] = offset[static_cast<int64_t>(h) * (a.ncells + 1) + g];
    if (o.mask) o.mask[hc] = 0;
}

// One wave per occupied compact slot: merged centroid = [C_0[l0] | C_1[l1] | ...].
__global__ __launch_bounds__(256) void ix_compact_merged_kernel(IxParams a, CompactOut o, const int32_t* n_active) {
    const int h = blockIdx.y;
    const int c = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (c >= min(n_active[h], o.n_c)) return;
    const int64_t hc = static_cast<int64_t>(h) * o.n_c + c;
    int64_t rem = o.gid[hc];
    int lab[4] = {0, 0, 0, 0};
    for (int p = a.P - 1; p >= 0; --p) {
        lab[p] = static_cast<int>(rem % a.k[p]);
        rem /= a.k[p];
    }
    for (int d = lane_id(); d < o.D; d += 64) {
        const int p = d / o.DP;
        o.merged[hc * o.D + d] =
            o.cent[((static_cast<int64_t>(h) * a.P + p) * a.kmax + lab[p]) * o.DP + (d - p * o.DP)];
    }
}

// Padding slots c >= n_active (and the closing offset).
__global__ __launch_bounds__(256) void ix_compact_pad_kernel(IxParams a, CompactOut o, const int32_t* n_active) {
    const int h = blockIdx.y;
    const int c = blockIdx.x * 256 + threadIdx.x;
    const int na = n_active[h];
    if (c == 0) o.offset[static_cast<int64_t>(h) * (o.n_c + 1) + o.n_c] = a.T;
    if (c >= o.n_c || c < na) return;
    const int64_t hc = static_cast<int64_t>(h) * o.n_c + c;
    o.gid[hc] = -1;
    o.size[hc] = 0;
    o.offset[static_cast<int64_t>(h) * (o.n_c + 1) + c] = a.T;
    if (o.mask) o.mask[hc] = 1;
    if (o.merged)
        for (int d = 0; d < o.D; ++d) o.merged[hc * o.D + d] = 0.0f;
}

// list[h][pos] = src[h][perm[h][pos]] for keys and values; 16 lanes per
// 256-byte row, 16 rows per wave with every load issued before any store.
// Loads and stores are non-temporal (each byte is touched once) and the
// loads unconditional (rows past T re-read token 0 and are not stored): 1.07
// GB per layer at configs[1] in ~150 us, against ~237 us with cached,
// predicated loads and stores.  (32 rows per wave, twice the loads in
// flight, ran at 3.1 TB/s even on the identity permutation.)
constexpr int kPermRowsPerWave = 16;
typedef unsigned int ix_u32x4_t __attribute__((ext_vector_type(4)));

__global__ __launch_bounds__(256) void ix_permute_kernel(const uint16_t* keys, const uint16_t* values, int64_t hs,
                                                         int64_t ts, int T, const int32_t* perm, uint16_t* lk,
                                                         uint16_t* lv, int64_t list_rows) {
    const int h = blockIdx.y;
    const int wave = threadIdx.x >> 6, lane = lane_id();
    const int rg = lane >> 4, li = lane & 15;
    const int base = (blockIdx.x * 4 + wave) * kPermRowsPerWave;
    const int my = base + lane;
    const int tok = (lane < kPermRowsPerWave && my < T) ? perm[static_cast<int64_t>(h) * T + my] : 0;
    constexpr int IT = kPermRowsPerWave / 4;
    ix_u32x4_t kv[IT], vv[IT];
#pragma unroll
    for (int it = 0; it < IT; ++it) {
        const int t = __shfl(tok, it * 4 + rg);
        const int64_t so = h * hs + static_cast<int64_t>(t) * ts + li * 8;
        kv[it] = __builtin_nontemporal_load(reinterpret_cast<const ix_u32x4_t*>(keys + so));
        vv[it] = __builtin_nontemporal_load(reinterpret_cast<const ix_u32x4_t*>(values + so));
    }
#pragma unroll
    for (int it = 0; it < IT; ++it) {
        const int pos = base + it * 4 + rg;
        if (pos < T) {
            const int64_t dofs = (static_cast<int64_t>(h) * list_rows + pos) * 128 + li * 8;
            __builtin_nontemporal_store(kv[it], reinterpret_cast<ix_u32x4_t*>(lk + dofs));
            __builtin_nontemporal_store(vv[it], reinterpret_cast<ix_u32x4_t*>(lv + dofs));
        }
    }
}

int validate(const imi_index_args* a, int& kmax, int64_t& ncells) {
    IMI_REQUIRE(a != nullptr, IMI_ERR_INVALID, "imi_build_index: null args");
    IMI_REQUIRE(a->keys && a->values && a->labels && a->cell_count && a->cell_offset && a->perm &&
                    a->list_keys && a->list_values,
                IMI_ERR_INVALID, "imi_build_index: null pointer argument");
    IMI_REQUIRE(a->kv_heads > 0 && a->n_tokens > 0, IMI_ERR_INVALID, "imi_build_index: empty input");
    IMI_REQUIRE(a->dim == 128, IMI_ERR_UNSUPPORTED, "imi_build_index: head_dim must be 128 (got %d)", a->dim);
    IMI_REQUIRE(a->parts == 1 || a->parts == 2 || a->parts == 4, IMI_ERR_UNSUPPORTED,
                "imi_build_index: parts must be 1 (IVF), 2 or 4");
    IMI_REQUIRE(a->list_rows >= a->n_tokens, IMI_ERR_INVALID, "imi_build_index: list_rows %lld < n_tokens %d",
                static_cast<long long>(a->list_rows), a->n_tokens);
    IMI_REQUIRE((a->token_stride % 8) == 0 && (a->head_stride % 8) == 0, IMI_ERR_INVALID,
                "imi_build_index: strides must be multiples of 8 elements");
    kmax = 0;
    ncells = 1;
    const int kcap = a->parts == 1 ? kIvfMaxK : kImiMaxK;
    for (int p = 0; p < a->parts; ++p) {
        IMI_REQUIRE(a->k[p] >= 1 && a->k[p] <= kcap, IMI_ERR_UNSUPPORTED, "imi_build_index: k[%d]=%d outside [1,%d]",
                    p, a->k[p], kcap);
        kmax = a->k[p] > kmax ? a->k[p] : kmax;
        ncells *= a->k[p];
    }
    IMI_REQUIRE(ncells <= (int64_t(1) << 26), IMI_ERR_UNSUPPORTED, "imi_build_index: %lld cells exceed 2^26",
                static_cast<long long>(ncells));
    const bool compact = a->compact_gid || a->compact_size || a->compact_offset || a->compact_centroids ||
                         a->compact_mask || a->n_active;
    if (compact) {
        IMI_REQUIRE(a->compact_gid && a->compact_size && a->compact_offset && a->n_active, IMI_ERR_INVALID,
                    "imi_build_index: compact gid, size, offset and n_active must be all set or all NULL");
        IMI_REQUIRE(!a->compact_centroids || a->centroids, IMI_ERR_INVALID,
                    "imi_build_index: merged compact centroids need the subspace centroids");
        const int64_t max_active = ncells < a->n_tokens ? ncells : a->n_tokens;
        IMI_REQUIRE(a->n_centroids >= max_active, IMI_ERR_INVALID,
                    "imi_build_index: n_centroids %d < possible occupied cells %lld", a->n_centroids,
                    static_cast<long long>(max_active));
    }
    return IMI_OK;
}

// tmp: the second token order and the two cell orders of the LSD passes
size_t workspace_bytes(const imi_index_args* a, int kmax, int64_t ncells, IxParams* p, int32_t* (*tmp)[3]) {
    const size_t items = static_cast<size_t>(a->kv_heads) * a->n_tokens;
    Carver cv(a->workspace);
    IxParams q{};
    superblocks(a->n_tokens, a->kv_heads, q.sbt, q.nsb);
    q.hist = cv.take<int32_t>(static_cast<size_t>(a->kv_heads) * kmax * q.nsb);
    q.cid = cv.take<int32_t>(static_cast<size_t>(a->kv_heads) * ncells);
    q.sums = cv.take<int32_t>(static_cast<size_t>(a->kv_heads) * 2 * ((ncells + kOffCells - 1) / kOffCells));
    int32_t* t[3];
    t[0] = cv.take<int32_t>(a->parts > 1 ? items : 1);
    t[1] = cv.take<int32_t>(items);
    t[2] = cv.take<int32_t>(a->parts > 1 ? items : 1);
    if (p) *p = q;
    if (tmp)
        for (int i = 0; i < 3; ++i) (*tmp)[i] = t[i];
    return cv.used();
}

uint32_t magic(uint32_t d) { return d > 1 ? static_cast<uint32_t>((uint64_t{1} << 32) / d + ((uint64_t{1} << 32) % d != 0)) : 0u; }

}  // namespace
}  // namespace imi

using namespace imi;

extern "C" int imi_index_workspace_size(const imi_index_args* a, size_t* bytes) {
    clear_error();
    int kmax;
    int64_t ncells;
    int rc = validate(a, kmax, ncells);
    if (rc) return rc;
    IMI_REQUIRE(bytes != nullptr, IMI_ERR_INVALID, "imi_index_workspace_size: null output");
    imi_index_args tmp = *a;
    tmp.workspace = nullptr;
    *bytes = workspace_bytes(&tmp, kmax, ncells, nullptr, nullptr);
    return IMI_OK;
}

extern "C" int imi_build_index(const imi_index_args* a, imi_stream_t stream_) {
    clear_error();
    hipStream_t stream = reinterpret_cast<hipStream_t>(stream_);
    int kmax;
    int64_t ncells;
    int rc = validate(a, kmax, ncells);
    if (rc) return rc;
    imi_index_args tmp = *a;
    tmp.workspace = nullptr;
    const size_t need = workspace_bytes(&tmp, kmax, ncells, nullptr, nullptr);
    IMI_REQUIRE(a->workspace != nullptr && a->workspace_bytes >= need, IMI_ERR_WORKSPACE,
                "imi_build_index: workspace %zu bytes < %zu required", a->workspace_bytes, need);
    IxParams p;
    int32_t* tmp_items[3];
    workspace_bytes(a, kmax, ncells, &p, &tmp_items);
    p.labels = a->labels;
    p.H = a->kv_heads;
    p.T = a->n_tokens;
    p.P = a->parts;
    p.kmax = kmax;
    for (int i = 0; i < 4; ++i) p.k[i] = i < a->parts ? a->k[i] : 1;
    p.ncells = ncells;
    const bool compact = a->compact_gid != nullptr;
    if (!compact) p.cid = nullptr;

    // LSD passes: last subspace first; the final pass lands in a->perm and
    // tmp_items[1] (the sorted cell ids).
    IxPass s{};
    const int waves = sort_waves(kmax);
    s.stage = p.sbt <= kStagedItems && place_lds_bytes(waves, kmax, p.sbt, true) <= 150 * 1024;
    const size_t lds = place_lds_bytes(waves, kmax, p.sbt, s.stage);
    if (lds > 64 * 1024)
        IMI_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(&ix_place_kernel),
                                          hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(lds)));
    uint32_t div = 1;
    for (int part = a->parts - 1; part >= 0; --part) {
        s.p = part;
        s.tok = s.tok_out;
        s.cell = s.cell_out;
        s.tok_out = part % 2 == 0 ? a->perm : tmp_items[0];
        s.cell_out = part % 2 == 0 ? tmp_items[1] : tmp_items[2];
        s.k = static_cast<uint32_t>(a->k[part]);
        s.div = div;
        s.div_magic = magic(s.div);
        s.k_magic = magic(s.k);
        div *= s.k;
        hipLaunchKernelGGL(ix_hist_kernel, dim3(p.nsb, p.H), dim3(64 * waves), s.k * sizeof(int), stream, p, s);
        IMI_LAUNCH_CHECK("ix_hist_kernel");
        hipLaunchKernelGGL(ix_scan_kernel, dim3(p.H), dim3(1024), 0, stream, p, static_cast<int>(s.k));
        IMI_LAUNCH_CHECK("ix_scan_kernel");
        hipLaunchKernelGGL(ix_place_kernel, dim3(p.nsb, p.H), dim3(64 * waves), lds, stream, p, s);
        IMI_LAUNCH_CHECK("ix_place_kernel");
    }

    const int64_t cells_total = ncells * p.H;
    hipLaunchKernelGGL(ix_zero_kernel, dim3(static_cast<unsigned>((cells_total + 255) / 256 < 65535 ? (cells_total + 255) / 256 : 65535)),
                       dim3(256), 0, stream, a->cell_count, cells_total);
    IMI_LAUNCH_CHECK("ix_zero_kernel");
    hipLaunchKernelGGL(ix_count_kernel, dim3((a->n_tokens + 255) / 256, p.H), dim3(256), 0, stream, p, tmp_items[1],
                       a->cell_count);
    IMI_LAUNCH_CHECK("ix_count_kernel");
    const int nchunk = static_cast<int>((ncells + kOffCells - 1) / kOffCells);
    hipLaunchKernelGGL(ix_chunk_sums_kernel, dim3(nchunk, p.H), dim3(256), 0, stream, p, a->cell_count, p.sums,
                       nchunk);
    IMI_LAUNCH_CHECK("ix_chunk_sums_kernel");
    hipLaunchKernelGGL(ix_offsets_kernel, dim3(nchunk, p.H), dim3(256), 0, stream, p, a->cell_count, a->cell_offset,
                       a->n_active, p.sums, nchunk);
    IMI_LAUNCH_CHECK("ix_offsets_kernel");

    if (compact) {
        CompactOut o;
        o.n_c = a->n_centroids;
        o.cent = a->centroids;
        o.D = a->dim;
        o.DP = a->dim / a->parts;
        o.gid = a->compact_gid;
        o.size = a->compact_size;
        o.offset = a->compact_offset;
        o.merged = a->compact_centroids;
        o.mask = a->compact_mask;
        hipLaunchKernelGGL(ix_compact_fill_kernel, dim3(static_cast<unsigned>((ncells + 255) / 256), p.H), dim3(256),
                           0, stream, p, o, a->cell_count, a->cell_offset);
        IMI_LAUNCH_CHECK("ix_compact_fill_kernel");
        if (o.merged) {
            hipLaunchKernelGGL(ix_compact_merged_kernel, dim3((o.n_c + 3) / 4, p.H), dim3(256), 0, stream, p, o,
                               a->n_active);
            IMI_LAUNCH_CHECK("ix_compact_merged_kernel");
        }
        hipLaunchKernelGGL(ix_compact_pad_kernel, dim3((o.n_c + 256) / 256, p.H), dim3(256), 0, stream, p, o,
                           a->n_active);
        IMI_LAUNCH_CHECK("ix_compact_pad_kernel");
    }

    hipLaunchKernelGGL(ix_permute_kernel, dim3((a->n_tokens + 4 * kPermRowsPerWave - 1) / (4 * kPermRowsPerWave), p.H),
                       dim3(256), 0, stream, a->keys,
                       a->values, a->head_stride, a->token_stride, a->n_tokens, a->perm, a->list_keys,
                       a->list_values, a->list_rows);
    IMI_LAUNCH_CHECK("ix_permute_kernel");
    return IMI_OK;
}
