// Per-(head, subspace) Lloyd k-means on gfx950.
//
// Reference: library/AdaptiveIMI/cpp_extensions/src/kmeans_core.cpp
//   distance     22-44   (8 FMA lanes, lane sums left to right)
//   E-step       222-242 (argmin, strict '<': lowest index wins ties)
//   early stop   244-262
//   M-step       265-312 (members summed in ascending token order, times
//                          1.0f/size; empty cluster <- x[uniform draw])
//   executor     384-501 (one independent run per (head, subspace))
//
// IVF (KmeansExecutorIVF, 503-595) is the one-subspace case: P = 1, Dp = 128,
// k up to kIvfMaxK, kmeans++ with seed 42.
//
// Work layout: every kernel covers all H*P (head, subspace) segments at once.
// E-step: distances are screened on the matrix cores (bf16 MFMA with the
// centroids split into hi + lo bf16 parts, under a proven rounding bound) and
// only the centroids that can still win get the exact reference distance.
// The member lists come from a stable counting sort per superblock of tokens;
// the M-step finds its members through every superblock's label offsets and
// sums each cluster sequentially in ascending token order (the reference's
// order with one thread per subspace run): one workgroup per cluster, one wave
// running the chains while three waves stream the member rows through
// register rings and an LDS hand-off.
#include <limits>
#include <random>
#include <type_traits>
#include <utility>
#include <vector>

#include "imi_common.hpp"
#include "imi_sort.hpp"

namespace imi {
namespace {

struct KmParams {
    const uint16_t* keys;
    int64_t hs, ts;
    int H, T, P, kmax, DP;
    int k[4];
    float* cent;       // [seg][kmax][DP]
    int32_t* labels;   // [seg][T]
    float* mind;       // [seg][T] or null
    float* wpart;      // [seg][4 nblk] inertia per 64 tokens, or null
    int32_t* sorted;   // [seg][T] member lists, superblock by superblock
    // [seg][nsb][kmax + 1] each superblock's first place of every label, then
    // its token count
    int32_t* loff;
    // [seg][kmax] ordinal of an empty cluster, otherwise -1, or -1 minus the size
    // of a cluster left to a workgroup (kWaveMost)
    int32_t* empties;
    float* prev;       // [seg][2] inertia of the last tested iteration
    int32_t* done;     // [seg] or null
    int32_t* iters;    // [seg] or null
    void* ppstats;     // kmeans++ block statistics, two launches' (init_mode 2)
    uint8_t *ppq, *ppqd;   // kmeans++ 8-bit copy, its dims' order, norms, scales, error bounds (or null)
    float *ppqn, *ppqs, *ppqe;
    int nblk;          // 256-token blocks
    int max_iters;
    float tol;
    int es_min;
    float es_rel;
    int exact;         // the E-step's distances are read (min distances or the early-stop inertia)
    int sbt;           // tokens per superblock of the member lists
    int nsb;           // superblocks per segment (at most kMaxSuper)
    float* ppmd;       // kmeans++: the second minima buffer [seg][T] (init_mode 2)
};

// The same distance with both rows read eight dims at a time (few registers).
template <int DP>
__device__ __forceinline__ float l2_lanes8_rolled(const uint16_t* x, const float* cr) {
    float acc[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) acc[j] = 0.0f;
#pragma unroll 2
    for (int i = 0; i < DP; i += 8) {
        const float4 c0 = *reinterpret_cast<const float4*>(cr + i);
        const float4 c1 = *reinterpret_cast<const float4*>(cr + i + 4);
        const uint4 v = *reinterpret_cast<const uint4*>(x + i);
        const float cv[8] = {c0.x, c0.y, c0.z, c0.w, c1.x, c1.y, c1.z, c1.w};
        const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const float d = (j & 1 ? bf16_hi(w[j / 2]) : bf16_lo(w[j / 2])) - cv[j];
            acc[j] = __builtin_fmaf(d, d, acc[j]);
        }
    }
    float t = acc[0];
#pragma unroll
    for (int j = 1; j < 8; ++j) t = t + acc[j];
    return t;
}

struct Draws {
    int32_t v[256];  // uniform draws for the empty clusters of one iteration
};

constexpr int kDraws = 256;      // empty-cluster draws one launch carries
constexpr int kIvfMaxK = 4096;   // IVF clusters per head

__global__ __launch_bounds__(64) void km_init_first_kernel(KmParams a) {
    const int c = blockIdx.x, seg = blockIdx.y;
    const int h = seg / a.P, p = seg % a.P;
    if (c >= a.k[p]) return;
    for (int d = threadIdx.x; d < a.DP; d += 64)
        a.cent[(static_cast<int64_t>(seg) * a.kmax + c) * a.DP + d] =
            bf16_to_f32(a.keys[h * a.hs + static_cast<int64_t>(c) * a.ts + p * a.DP + d]);
}

// Reference distance between a row in its bf16 load registers (each 16-byte
// part holds dims i .. i+7 of lanes 0..7) and the fp32 row cr: lane j
// accumulates dims j, j+8, ... with fused multiply-add, then the eight lane
// sums are added left to right.
template <int DP, typename V>
__device__ __forceinline__ float l2_lanes8_bf16(const V (&v)[DP / 8], const float* cr) {
    float acc[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) acc[j] = 0.0f;
#pragma unroll
    for (int i = 0; i < DP / 8; ++i) {
        const float4 c0 = *reinterpret_cast<const float4*>(cr + 8 * i);
        const float4 c1 = *reinterpret_cast<const float4*>(cr + 8 * i + 4);
        float d;
        d = bf16_lo(v[i].x) - c0.x; acc[0] = __builtin_fmaf(d, d, acc[0]);
        d = bf16_hi(v[i].x) - c0.y; acc[1] = __builtin_fmaf(d, d, acc[1]);
        d = bf16_lo(v[i].y) - c0.z; acc[2] = __builtin_fmaf(d, d, acc[2]);
        d = bf16_hi(v[i].y) - c0.w; acc[3] = __builtin_fmaf(d, d, acc[3]);
        d = bf16_lo(v[i].z) - c1.x; acc[4] = __builtin_fmaf(d, d, acc[4]);
        d = bf16_hi(v[i].z) - c1.y; acc[5] = __builtin_fmaf(d, d, acc[5]);
        d = bf16_lo(v[i].w) - c1.z; acc[6] = __builtin_fmaf(d, d, acc[6]);
        d = bf16_hi(v[i].w) - c1.w; acc[7] = __builtin_fmaf(d, d, acc[7]);
    }
    float t = acc[0];
#pragma unroll
    for (int j = 1; j < 8; ++j) t = t + acc[j];
    return t;
}

// ------------------------------------------------------------------ E-step
// Matrix-core screening for any k.  With the mean of the segment's first and
// middle centroid as the origin m (subspaces; m = 0 for IVF) and c' = c - m, the
// value
//   f(c) = x.c' - (m.c' + |c'|^2 / 2) = (|x - m|^2 - D(x, c)) / 2
// orders the centroids like the distance (largest f first), and its terms
// don't grow with a common offset of keys and centroids beyond the first
// power.  x.c' runs on v_mfma_f32_16x16x32_bf16: x is bf16 already and c'
// enters as two bf16 parts (hi = bf16(c'), lo = bf16(c' - hi)); the
// accumulators start at the second term.  Rounding analysis with C = max|c'|,
// N = |x|^2 + |m|^2 and R = sqrt(2 N) C + C^2 / 2, which bounds every partial
// sum of f.  Relative to R: 2 DP accumulations of at most 2^-23 each (also if
// the matrix core truncates), the split of c' (two round-to-nearest bf16 steps:
// 2^-18), the second term's chains (DP / 4 + 4 operations of 2^-24), the
// rounding of c' itself (2^-23): 3.63e-5, 2.04e-5 and 1.23e-5 for 128, 64 and
// 32 dims, and twice that (e_sum, with 5 %) between two centroids.  The
// reference's own distance is off by at most (DP / 8 + 9) 2^-24 of D (8 FMA
// chains + 7 adds, the square of a rounded difference); the best centroid's D
// is at most 2 (N + C^2): e_ref (N + C^2).
//
// Each lane keeps the three largest f of its token (a max and two med3 per
// value), each value carrying its centroid's number in its lowest bits, which
// moves a value by less than 2^(bits - 23) of it; for IVF the number inside its
// chunk of 64, the chunk beside it.  So the reference's winner has f >= best - E,
//   E = e_sum R + 2^(bits - 22) |best| + e_ref (N + C^2) + 1e-30
// (the last term for subnormals):
//   second < best - E   the best is the reference's label;
//   third < best - E    best and second get the exact reference distance
//                       (l2 in 8 lanes, strict '<' over ascending c);
//   otherwise, for equal best and second values (IVF: their chunks cannot be
//   told apart) and for non-finite or huge magnitudes (N + C^2 > 1e37), the
//   token is undecided.  Up to kFewTokens undecided tokens of a wave get every
//   centroid's distance one token at a time.  More of them: the block is
//   screened again, the centroids that reach each token's bound are queued
//   and get the distance, 64 pairs at a time; where they are more than k / 4
//   per token, where magnitudes are huge, and for IVF, every lane goes
//   through all centroids for its token (nearest_of_all).
// With k-means centroids over the benchmark's keys 0.5-1 % of the tokens take
// the second form and 0.01 % the third (k = 32..1018).  Outputs (labels, min
// distances, inertia partials) are those of the exhaustive loop.
//
// The origin and the queue matter for keys unlike those.  Lloyd over 8 x 128k
// keys of N(0, 1), k = 64, 10 iterations, and k = 181, 6 iterations, with the
// bound in |x|^2 + max|c|^2 and every centroid for each undecided token ->
// now: four channels of mean 30: 10.6 -> 1.40 and 22.6 -> 1.36 ms; means of
// deviation 10: 22.9 -> 1.49 and 41.7 -> 1.62 ms, of 100: 27.9 -> 8.4 and
// 47.6 -> 6.8; 60 % of the keys within 0.05 of one: 21.3 -> 4.2 and 35.7 ->
// 4.2; row lengths log-normal: 28.4 -> 7.3 and 46.2 -> 8.4.  IVF, 16k, k =
// 1018, 10 iterations: means of deviation 10: 35.4 -> 10.9 ms (8 x 16k x
// 1018 distances in 1 ms).
//
// A wave owns 64 tokens (four 16-token tiles) and shares nothing with the
// other waves but the packed centroids, so the loop over its token blocks has
// no barrier and the waves' loads, matrix work and re-checks overlap; each
// block's tokens are loaded while the one before is re-checked.  The
// centroids are packed into LDS in the matrix-core operand layout by the
// workgroup: all of them at once for subspaces (4 DP bytes each), in double-
// buffered chunks of 64 for IVF (STREAM; an origin would cost it 11 % on the
// benchmark's keys, since every block of tokens packs the centroids again).
//
// Bound by: reading the keys up to k = 64 (64 x 64, 128k tokens, 8 heads: 268
// MB in 60 us, 4.5 TB/s; a barrier-synchronised form with the label ranks in
// it took 85 us), the three VALU operations and the and-or per value beside
// the matrix work beyond (k = 181, 512k tokens: 490 us; 4.65 ms as fp32
// distances to every centroid; IVF, k = 1018, 16k tokens, 8 heads: 104 us,
// 1.02 ms as such).
typedef __attribute__((ext_vector_type(8))) __bf16 km_bf16x8_t;
typedef __attribute__((ext_vector_type(4))) float km_f32x4_t;
typedef __attribute__((ext_vector_type(4))) unsigned int km_u32x4_t;
typedef __attribute__((ext_vector_type(2))) unsigned int km_u32x2_t;
typedef __attribute__((ext_vector_type(4))) short km_s16x4_t;
typedef __attribute__((address_space(3))) km_s16x4_t km_lds_s16x4_t;

constexpr float kFltMax = 3.402823466e38f;
constexpr int kChunkTiles = 4;   // 16-centroid tiles per streamed chunk

// Distances the E-step has to produce: none (labels only), exact ones with
// the fp32 centroid rows in LDS, or with the rows in global memory.
enum KmExact { kLabelsOnly = 0, kExactLds = 1, kExactGlobal = 2 };

// Row shift left by K inside a row of 16 lanes: lane i gets lane i + K's value.
template <int K>
__device__ __forceinline__ float dpp_row_shl(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x100 + K, 0xF, 0xF, false));
}

// Two fp32 values rounded to bf16 (nearest even), packed (v_cvt_pk_bf16_f32).
__device__ __forceinline__ uint32_t pack_bf16(float a, float b) {
    typedef __attribute__((ext_vector_type(2))) float f2;
    typedef __attribute__((ext_vector_type(2))) __bf16 b2;
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(f2{a, b}, b2));
}

// max without the operand canonicalisation fmaxf costs (one more VALU
// operation per screened value); no operand is a signalling NaN that matters:
// NaN magnitudes send the token through every centroid.
__device__ __forceinline__ float max_raw(float a, float b) {
    float r;
    asm("v_max_f32 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
}

// One lane's share of a 16-centroid tile: dims 32 kh + 8 (lane / 16) .. + 7 of
// centroid 16 ct + lane % 16, less the origin's (ORIGIN: half of org), as hi
// and lo bf16 operands; sq += the dims' squares, dot += their products with org.
template <bool ORIGIN>
__device__ __forceinline__ void pack_centroid(const float4 (&c)[2], const float4* org, km_u32x4_t& hi, km_u32x4_t& lo,
                                              float& sq, float& dot) {
    float v[8] = {c[0].x, c[0].y, c[0].z, c[0].w, c[1].x, c[1].y, c[1].z, c[1].w};
    if constexpr (ORIGIN) {
        const float m[8] = {org[0].x, org[0].y, org[0].z, org[0].w, org[1].x, org[1].y, org[1].z, org[1].w};
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            v[i] = __builtin_fmaf(-0.5f, m[i], v[i]);
            dot = __builtin_fmaf(v[i], m[i], dot);
        }
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const uint32_t h = pack_bf16(v[2 * i], v[2 * i + 1]);
        hi[i] = h;
        lo[i] = pack_bf16(v[2 * i] - bf16_lo(h), v[2 * i + 1] - bf16_hi(h));
        sq = __builtin_fmaf(v[2 * i], v[2 * i], sq);
        sq = __builtin_fmaf(v[2 * i + 1], v[2 * i + 1], sq);
    }
}

// The three largest values of a token (best >= second >= third).
struct Top3 {
    float b, s, t;
    __device__ __forceinline__ void add(float v) {
        t = __builtin_amdgcn_fmed3f(s, t, v);
        s = __builtin_amdgcn_fmed3f(b, s, v);
        b = max_raw(b, v);
    }
    __device__ __forceinline__ void merge(const Top3& o) {
        add(o.b);
        add(o.s);
        add(o.t);
    }
};

// permlane swaps of two values: after swap32 the lanes below 32 hold x of both
// halves (x, y) and the others y of both halves; swap16 does so for the even
// and odd rows of 16 lanes.
__device__ __forceinline__ void swap32(float& x, float& y) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(y), false, false);
    x = __uint_as_float(r[0]);
    y = __uint_as_float(r[1]);
}
__device__ __forceinline__ void swap16(float& x, float& y) {
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(y), false, false);
    x = __uint_as_float(r[0]);
    y = __uint_as_float(r[1]);
}
// Three largest values with the centroids of the first two (STREAM: a value
// carries only its number in the chunk).
struct Top3Ids {
    Top3 v;
    int ib, is;
};

// Halves (or rows) exchange their tiles: the lanes that keep x's tile get y's
// lanes' part of it, the others x's lanes' part of y's tile.
template <bool HALF, bool IDS>
__device__ __forceinline__ Top3Ids swap_merge(Top3Ids x, Top3Ids y) {
    auto swap = [](float& p, float& q) {
        if (HALF)
            swap32(p, q);
        else
            swap16(p, q);
    };
    swap(x.v.b, y.v.b);
    swap(x.v.s, y.v.s);
    swap(x.v.t, y.v.t);
    if (IDS) {
        float xi = __int_as_float(x.ib), yi = __int_as_float(y.ib), xj = __int_as_float(x.is), yj = __int_as_float(y.is);
        swap(xi, yi);
        swap(xj, yj);
        x.ib = __float_as_int(xi);
        x.is = __float_as_int(xj);
        y.ib = __float_as_int(yi);
        y.is = __float_as_int(yj);
        const bool xb = x.v.b >= y.v.b;
        const bool keep = xb ? x.v.s >= y.v.b : y.v.s >= x.v.b;   // the winner's second stays second
        const int ib = xb ? x.ib : y.ib;
        x.is = xb ? (keep ? x.is : y.ib) : (keep ? y.is : x.ib);
        x.ib = ib;
    }
    x.v.merge(y.v);
    return x;
}

// The value, computed where it is used: what depends on it isn't kept in
// registers over the loop around a seldom taken branch.
__device__ __forceinline__ int opaque(int v) {
    asm volatile("" : "+v"(v));
    return v;
}

// Tokens of a wave up to which the exhaustive form takes them one by one, its
// lanes over the centroids; beyond, every lane takes its own token.
constexpr int kFewTokens = 8;

// The exhaustive form for a wave's 64 tokens, all lanes active: each lane has
// its token's widened row; a centroid is spread over every row of 16 lanes
// (lane q: dims DP / 16 q ..) and broadcast as an operand modifier of the
// subtraction (row_newbcast), so a dim takes two VALU operations and no load.
// The next centroid's part is loaded meanwhile.  (c - x) has the square of
// (x - c).
template <int K>
__device__ __forceinline__ float row_bcast(float v) {
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x150 + K, 0xF, 0xF, true));
}

template <int DP, int... I>
__device__ __forceinline__ float l2_lanes8_spread(const float (&x)[DP], const float (&c)[DP / 16],
                                                  std::integer_sequence<int, I...>) {
    float acc[8] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
    const auto dim = [&](auto i) {
        constexpr int N = decltype(i)::value;
        const float d = row_bcast<N / (DP / 16)>(c[N % (DP / 16)]) - x[N];
        acc[N % 8] = __builtin_fmaf(d, d, acc[N % 8]);
    };
    (dim(std::integral_constant<int, I>{}), ...);
    float t = acc[0];
#pragma unroll
    for (int j = 1; j < 8; ++j) t = t + acc[j];
    return t;
}

template <int DP>
__device__ __forceinline__ void load_spread(const float* row, int q, float (&c)[DP / 16]) {
#pragma unroll
    for (int e = 0; e < DP / 16; e += 2) {
        const float2 v = *reinterpret_cast<const float2*>(row + DP / 16 * q + e);
        c[e] = v.x;
        c[e + 1] = v.y;
    }
}

// Smallest distance of the lane's row and the lowest centroid that has it.
template <int DP>
__device__ __forceinline__ void nearest_of_all(const uint16_t* row, const float* cg, int k, float& best, int& arg) {
    float x[DP];
#pragma unroll
    for (int i = 0; i < DP / 8; ++i) {
        const km_u32x4_t v = reinterpret_cast<const km_u32x4_t*>(row)[i];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            x[8 * i + 2 * e] = bf16_lo(v[e]);
            x[8 * i + 2 * e + 1] = bf16_hi(v[e]);
        }
    }
    best = kFltMax;
    arg = 0;
    float next[DP / 16];
    const int q = opaque(lane_id()) & 15;
    load_spread<DP>(cg, q, next);
#pragma unroll 1
    for (int c = 0; c < k; ++c) {
        float cv[DP / 16];
#pragma unroll
        for (int e = 0; e < DP / 16; ++e) cv[e] = next[e];
        load_spread<DP>(cg + static_cast<int64_t>(min(c + 1, k - 1)) * DP, q, next);
        __builtin_amdgcn_sched_barrier(0);   // above the chains, its wait below them
        const float d = l2_lanes8_spread<DP>(x, cv, std::make_integer_sequence<int, DP>{});
        // (loaded here, not where the next step uses the values)
#pragma unroll
        for (int e = 0; e < DP / 16; ++e) asm volatile("" : "+v"(next[e]));
        if (d < best) {
            best = d;
            arg = c;
        }
    }
}

template <int DP>
struct ScreenLds {
    static constexpr int KH = DP / 32;
    static size_t packed(int tiles) { return static_cast<size_t>(tiles) * (KH * 2 * 64 * 16 + 64); }
    static size_t rows(int kmax) { return static_cast<size_t>(kmax) * (DP + 4) * sizeof(float); }
};

template <int DP, int NW, bool STREAM, int EXACT>
__global__ __launch_bounds__(64 * NW, (STREAM || EXACT == kExactGlobal ? 2 : EXACT ? 3 : DP == 32 ? 5 : 4)) void km_screen_kernel(KmParams a, int chunks) {
    constexpr int KH = DP / 32;   // 32-dim K steps per subvector
    constexpr int CS = DP + 4;    // padded fp32 row
    constexpr bool ORIGIN = !STREAM;
    extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];
    const int seg = blockIdx.y;
    if (a.done && a.done[seg]) return;
    const int h = seg / a.P, p = seg % a.P;
    const int k = a.k[p];
    const int nct = (k + 15) >> 4;
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int grp = lane >> 4;
    // packed tiles [tile][KH][hi, lo][64 lanes], then f's second term [tile][16]
    const int tiles = STREAM ? 2 * kChunkTiles : nct;
    km_u32x4_t* apk = reinterpret_cast<km_u32x4_t*>(smem_raw);
    float* cch = reinterpret_cast<float*>(apk + tiles * KH * 2 * 64);
    float* cs = cch + tiles * 16;   // [k][CS] (kExactLds)
    const float* cg = a.cent + static_cast<int64_t>(seg) * a.kmax * DP;
    const uint16_t* kb = a.keys + h * a.hs + p * DP;
    // bits of the centroid number a value carries (of its number in the chunk)
    const int nbits = STREAM ? bits_for(16 * kChunkTiles) : bits_for(nct * 16);
    const uint32_t idx_mask = ~((1u << nbits) - 1u);
    constexpr float e_ref = DP == 128 ? 0x1.ap-19f : DP == 64 ? 0x1.2p-19f : 0x1.bp-20f;
    constexpr float e_sum = DP == 128 ? 0x1.4p-14f : DP == 64 ? 0x1.7p-15f : 0x1.bp-16f;
    const float e_num = ldexpf(1.0f + 0x1p-10f, nbits - 22);
    // the lane's rows of a 16-token tile
    const uint16_t* lane_rows = kb + static_cast<int64_t>(lane & 15) * a.ts + 8 * grp;
    float ccmax = 0.0f;   // largest |c - m|^2: of the lane's own centroids until the reduction
    float mm = 0.0f;      // |m|^2
    // what E takes from the centroids: the factor of sqrt(N), the terms of C
    // alone, the factor of |best|; C^2 (read where they are used: in registers
    // they would spill)
    __shared__ float4 s_bound[1];

    // tile ct -> slot: one wave packs it; padding centroids are zero rows
    // whose f stays at -3e38
    auto load_tile = [&](int ct, float4 (&v)[2 * KH]) {
        const int c = min(16 * ct + (lane & 15), k - 1);
        const float4* row = reinterpret_cast<const float4*>(cg + static_cast<int64_t>(c) * DP);
#pragma unroll
        for (int kh = 0; kh < KH; ++kh) {
            v[2 * kh] = row[8 * kh + 2 * grp];
            v[2 * kh + 1] = row[8 * kh + 2 * grp + 1];
        }
    };
    auto store_tile = [&](int ct, int slot, float4 (&v)[2 * KH], const float4* org) {
        const bool real = 16 * ct + (lane & 15) < k;
        float sq = 0.0f, dot = 0.0f;
#pragma unroll
        for (int kh = 0; kh < KH; ++kh) {
            km_u32x4_t hi, lo;
            const float4 part[2] = {v[2 * kh], v[2 * kh + 1]};
            pack_centroid<ORIGIN>(part, org + 2 * kh, hi, lo, sq, dot);
            const km_u32x4_t zero = km_u32x4_t{0u, 0u, 0u, 0u};
            apk[((slot * KH + kh) * 2 + 0) * 64 + lane] = real ? hi : zero;
            apk[((slot * KH + kh) * 2 + 1) * 64 + lane] = real ? lo : zero;
        }
        sq += xor16(sq);
        sq += xor32(sq);
        if constexpr (ORIGIN) {
            dot += xor16(dot);
            dot += xor32(dot);
        }
        if (real) ccmax = sq > ccmax || sq != sq ? sq : ccmax;   // a NaN norm stays
        if (lane < 16) cch[slot * 16 + lane] = real ? -0.5f * (sq + dot) : -3e38f;
    };
    auto reduce_ccmax = [&](float* sh) {
        // (fmax would drop a NaN: an infinite bound stands for it)
        float m = ccmax == ccmax ? ccmax : INFINITY;
        m = wave_max(m);
        if (lane == 0) sh[wave] = m;
        __syncthreads();
        m = sh[0];
#pragma unroll
        for (int w = 1; w < NW; ++w) m = fmaxf(m, sh[w]);
        ccmax = m;
        // (every wave writes the values it reads)
        s_bound[0] = make_float4(e_sum * 1.4142137f * __builtin_amdgcn_sqrtf(m), (0.5f * e_sum + e_ref) * m + 1e-30f, e_num, m);
        wave_lds_order();
    };
    const int nblk = (a.T + 64 * NW - 1) / (64 * NW);
    const int blk0 = blockIdx.x * chunks, blk1 = min(blk0 + chunks, nblk);
    // B operands of the wave's four 16-token tiles of block blk (lane l: token
    // l % 16, dims 32 kh + 8 (l / 16) .. + 7); tokens past T re-read token T - 1
    km_u32x4_t bq[4][KH];
    auto load_tokens = [&](int blk) {
        const int t0 = __builtin_amdgcn_readfirstlane((blk * NW + wave) * 64);
        const uint16_t* src[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) src[j] = lane_rows + static_cast<int64_t>(t0 + 16 * j) * a.ts;
        if (t0 + 64 > a.T) {
            const int l = opaque(lane);
#pragma unroll
            for (int j = 0; j < 4; ++j)
                src[j] = kb + static_cast<int64_t>(min(t0 + 16 * j + (l & 15), a.T - 1)) * a.ts + 8 * (l >> 4);
        }
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int kh = 0; kh < KH; ++kh) bq[j][kh] = *reinterpret_cast<const km_u32x4_t*>(src[j] + kh * 32);
    };
    // the first block's tokens come while the centroids are packed, each
    // later block's while the one before is re-checked and stored
    load_tokens(blk0);
    __shared__ float s_cc[NW];
    // (distance, centroid) of a wave's tokens and its queue of (token, centroid)
    // pairs (more than one centroid reaches the bound of many tokens)
    __shared__ unsigned long long s_won[STREAM ? 1 : NW][64];
    __shared__ uint16_t s_pairs[STREAM ? 1 : NW][128];
    if constexpr (!STREAM) {
        float4 org[2 * KH], far[2 * KH];
        const float4* row0 = reinterpret_cast<const float4*>(cg);
        const float4* row1 = reinterpret_cast<const float4*>(cg + static_cast<int64_t>(k / 2) * DP);
#pragma unroll
        for (int i = 0; i < 2 * KH; ++i) {
            org[i] = row0[8 * (i / 2) + 2 * grp + i % 2];
            far[i] = row1[8 * (i / 2) + 2 * grp + i % 2];
        }
#pragma unroll
        for (int i = 0; i < 2 * KH; ++i)
            org[i] = make_float4(org[i].x + far[i].x, org[i].y + far[i].y, org[i].z + far[i].z, org[i].w + far[i].w);
        for (int ct = wave; ct < nct; ct += NW) {
            float4 v[2 * KH];
            load_tile(ct, v);
            store_tile(ct, ct, v, org);
        }
#pragma unroll
        for (int i = 0; i < 2 * KH; ++i) {
            mm = __builtin_fmaf(org[i].x, org[i].x, mm);
            mm = __builtin_fmaf(org[i].y, org[i].y, mm);
            mm = __builtin_fmaf(org[i].z, org[i].z, mm);
            mm = __builtin_fmaf(org[i].w, org[i].w, mm);
        }
        mm += xor16(mm);
        mm += xor32(mm);
        mm = 0.25f * __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(mm)));
        if constexpr (EXACT == kExactLds) {
            for (int i = tid; i < k * (DP / 4); i += 64 * NW)
                *reinterpret_cast<float4*>(cs + (i / (DP / 4)) * CS + 4 * (i % (DP / 4))) =
                    reinterpret_cast<const float4*>(cg)[i];
        }
        reduce_ccmax(s_cc);
    }

#pragma unroll 1
    for (int blk = blk0; blk < blk1; ++blk) {
        const int t0 = __builtin_amdgcn_readfirstlane((blk * NW + wave) * 64);
        if (!STREAM && t0 >= a.T) break;   // (streaming waves keep to the barriers)
        const int t = t0 + lane;
        const bool valid = t < a.T;
        Top3 top[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) top[j] = Top3{-INFINITY, -INFINITY, -INFINITY};
        // centroid numbers of the lane's four accumulator rows (kept apart, so
        // that the number enters a value with one and-or)
        uint32_t num[4];
        auto number_from = [&](uint32_t c) {
#pragma unroll
            for (uint32_t r = 0; r < 4; ++r) {
                num[r] = c + 4 * grp + r;
                asm("" : "+v"(num[r]));
            }
        };
        number_from(0);
        // f of the 16 centroids of packed slot `slot`, and the largest three with it
        typedef km_f32x4_t Acc[4];
        auto products = [&](int slot, Acc& acc) {
            const km_f32x4_t init = *reinterpret_cast<const km_f32x4_t*>(cch + slot * 16 + 4 * grp);
#pragma unroll
            for (int j = 0; j < 4; ++j) acc[j] = init;
#pragma unroll
            for (int kh = 0; kh < KH; ++kh)
#pragma unroll
                for (int part = 0; part < 2; ++part) {
                    const km_bf16x8_t c =
                        __builtin_bit_cast(km_bf16x8_t, apk[((slot * KH + kh) * 2 + part) * 64 + lane]);
#pragma unroll
                    for (int j = 0; j < 4; ++j)
                        acc[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(c, __builtin_bit_cast(km_bf16x8_t, bq[j][kh]),
                                                                         acc[j], 0, 0, 0);
                }
        };
        auto largest = [&](const Acc& acc) {
#pragma unroll
            for (int r = 0; r < 4; ++r)
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    top[j].add(__uint_as_float((__float_as_uint(acc[j][r]) & idx_mask) | num[r]));
#pragma unroll
            for (int r = 0; r < 4; ++r) num[r] += 16;
        };
        // `n` tiles from slot s0 on: a tile's products run beside the comparisons
        // of the tile before (one matrix operation, then its share of VALU; 59.4
        // against 62.7 us at k = 64, 128k tokens, 485 against 501 at k = 181, 512k)
        auto overlap = [&]() {
#pragma unroll
            for (int i = 0; i < 8 * KH; ++i) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x002, 4, 0);
            }
        };
        auto screen_tiles = [&](int s0, int n) {
            Acc x, y;
            // (128 dims: the tokens take the registers of a second tile; 32 dims:
            // measured slower, 144 against 135 us for the 4-way index at 256k)
            if (DP != 64) {
#pragma unroll 1
                for (int i = 0; i < n; ++i) {
                    products(s0 + i, x);
                    largest(x);
                }
                return;
            }
            products(s0, x);
            int i = 1;
#pragma unroll 1
            for (; i + 1 < n; i += 2) {
                products(s0 + i, y);
                largest(x);
                overlap();
                products(s0 + i + 1, x);
                largest(y);
                overlap();
            }
            if (i < n) {
                products(s0 + i, y);
                largest(x);
                overlap();
                largest(y);
            } else {
                largest(x);
            }
        };
        int chb[4] = {0, 0, 0, 0}, chs[4] = {0, 0, 0, 0};   // chunks of best and second (STREAM)
        if constexpr (STREAM) {
            // chunk q in slots kChunkTiles (q % 2) ..: wave w packs its tile
            // w of chunk q + 1 while chunk q is screened
            static_assert(!STREAM || NW == kChunkTiles, "one tile per wave and chunk");
            const int nch = (nct + kChunkTiles - 1) / kChunkTiles;
            float4 v[2 * KH];
            load_tile(wave, v);
            __syncthreads();   // the previous block's reads are done
            store_tile(wave, wave, v, v);
            __syncthreads();
#pragma unroll 1
            for (int q = 0; q < nch; ++q) {
                const int nxt = (q + 1) * kChunkTiles + wave;
                if (q + 1 < nch) load_tile(nxt, v);
                float pb[4], ps[4];
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    pb[j] = top[j].b;
                    ps[j] = top[j].s;
                }
                number_from(0);
                screen_tiles((q & 1) * kChunkTiles, kChunkTiles);
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    if (top[j].s != ps[j]) chs[j] = top[j].s == pb[j] ? chb[j] : q;
                    if (top[j].b != pb[j]) chb[j] = q;
                }
                if (q + 1 < nch) store_tile(nxt, ((q + 1) & 1) * kChunkTiles + wave, v, v);
                __syncthreads();
            }
            if (blk == blk0) reduce_ccmax(s_cc);
        } else {
            screen_tiles(0, nct);
        }
        // |x|^2: each lane has its quarter of every tile's dims
        float xs[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            xs[j] = 0.0f;
#pragma unroll
            for (int kh = 0; kh < KH; ++kh)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    typedef __attribute__((ext_vector_type(2))) __bf16 b2;
                    const b2 x2 = __builtin_bit_cast(b2, static_cast<uint32_t>(bq[j][kh][i]));
                    xs[j] = __builtin_amdgcn_fdot2_f32_bf16(x2, x2, xs[j], false);
                }
        }
        // row g of the wave ends with tile g: halves exchange tiles (0, 2) and
        // (1, 3), then rows
        swap32(xs[0], xs[2]);
        swap32(xs[1], xs[3]);
        float x02 = xs[0] + xs[2], x13 = xs[1] + xs[3];
        swap16(x02, x13);
        const float4 e = s_bound[opaque(0)];
        const float norms = (x02 + x13) + mm;
        Top3Ids own[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            own[j].v = top[j];
            own[j].ib = 16 * kChunkTiles * chb[j] + static_cast<int>(__float_as_uint(top[j].b) & ~idx_mask);
            own[j].is = 16 * kChunkTiles * chs[j] + static_cast<int>(__float_as_uint(top[j].s) & ~idx_mask);
        }
        const Top3Ids m02 = swap_merge<true, STREAM>(own[0], own[2]);
        const Top3Ids m13 = swap_merge<true, STREAM>(own[1], own[3]);
        const Top3Ids mi = swap_merge<false, STREAM>(m02, m13);
        const Top3 m = mi.v;
        const float lim = m.b - ((e.x * __builtin_amdgcn_sqrtf(norms) + e.y) + (e.z * fabsf(m.b) + e_ref * norms));
        const bool wild = !(norms + e.w <= 1e37f);
        const bool every = wild || !(m.t < lim) || m.s == m.b;
        const bool pair = !every && !(m.s < lim);
        const int c1 = STREAM ? mi.ib : static_cast<int>(__float_as_uint(m.b) & ~idx_mask);
        const int c2 = STREAM ? mi.is : static_cast<int>(__float_as_uint(m.s) & ~idx_mask);
        float best = kFltMax;
        int arg = 0;
        // every centroid: a few tokens spread over the lanes by centroid, or
        // each token on its own lane
        uint64_t full = __ballot(every && valid);
        if (full) {
            if (__popcll(full) > kFewTokens) {
                bool found = false;
                const int fl = opaque(lane), fw = opaque(wave);
                if constexpr (!STREAM) {
                    // the block is screened again: the centroids that reach a
                    // token's bound are counted and, where they are few, get
                    // the exact distance, 64 (token, centroid) pairs at a time
                    float lims[4];
#pragma unroll
                    for (int j = 0; j < 4; ++j)
                        lims[j] = __shfl(every && valid ? lim : INFINITY, 16 * j + (fl & 15));
                    auto reaching = [&](int ct) {
                        Acc acc;
                        products(ct, acc);
                        uint32_t mask = 0;   // bit 4 j + r
#pragma unroll
                        for (int j = 0; j < 4; ++j)
#pragma unroll
                            for (int r = 0; r < 4; ++r) mask |= acc[j][r] >= lims[j] ? 1u << (4 * j + r) : 0u;
                        return mask;
                    };
                    int pairs = 0;
#pragma unroll 1
                    for (int i = 0; i < nct; ++i) pairs += __popc(reaching(i));
                    if (__ballot(every && valid && wild) == 0 && wave_sum_i(pairs) <= 16 * k) {
                        s_won[fw][fl] = ~0ull;
                        auto settle = [&](int n) {   // the queue's first n pairs
                            wave_lds_order();
                            if (fl < n) {
                                const int code = s_pairs[fw][fl], tk = code >> 9, c = code & 511;
                                const float d = l2_lanes8_rolled<DP>(kb + static_cast<int64_t>(t0 + tk) * a.ts,
                                                                     cg + static_cast<int64_t>(c) * DP);
                                if (d < kFltMax)
                                    atomicMin(&s_won[fw][tk], (static_cast<unsigned long long>(__float_as_uint(d)) << 32) |
                                                                    static_cast<uint32_t>(c));
                            }
                        };
                        int nq = 0;
#pragma unroll 1
                        for (int i = 0; i < nct; ++i) {
                            uint32_t mask = reaching(i);
#pragma unroll 1
                            while (const uint64_t has = __ballot(mask != 0)) {
                                if (mask != 0) {
                                    const int b = __builtin_ctz(mask);
                                    mask &= mask - 1;
                                    s_pairs[fw][nq + __builtin_amdgcn_mbcnt_hi(static_cast<uint32_t>(has >> 32), __builtin_amdgcn_mbcnt_lo(static_cast<uint32_t>(has), 0u))] = static_cast<uint16_t>(
                                        (16 * (b >> 2) + (fl & 15)) << 9 | (16 * i + 4 * (fl >> 4) + (b & 3)));
                                }
                                nq += __popcll(has);
                                if (nq < 64) continue;
                                settle(64);
                                nq -= 64;
                                const uint16_t rest = s_pairs[fw][64 + fl];
                                wave_lds_order();
                                s_pairs[fw][fl] = rest;
                            }
                        }
                        settle(nq);
                        wave_lds_order();
                        found = true;
                        const unsigned long long key = s_won[fw][fl];
                        if (every && key != ~0ull) {
                            arg = static_cast<int>(static_cast<uint32_t>(key));
                            best = __uint_as_float(static_cast<uint32_t>(key >> 32));
                        }
                    }
                }
                if (!found) {
                    float d;
                    int at;
                    nearest_of_all<DP>(kb + static_cast<int64_t>(min(t0 + fl, a.T - 1)) * a.ts, cg, k, d, at);
                    if (every) {
                        best = d;
                        arg = at;
                    }
                }
            } else {
                while (full) {
                    const int tk = __builtin_ctzll(full);
                    full &= full - 1;
                    const uint16_t* row = kb + static_cast<int64_t>(t0 + tk) * a.ts;
                    unsigned long long key = ~0ull;
#pragma unroll 1
                    for (int c = opaque(lane); c < k; c += 64) {
                        const float d = l2_lanes8_rolled<DP>(row, cg + static_cast<int64_t>(c) * DP);
                        const unsigned long long kv =
                            (static_cast<unsigned long long>(__float_as_uint(d)) << 32) | static_cast<uint32_t>(c);
                        if (d < kFltMax && kv < key) key = kv;
                    }
#pragma unroll
                    for (int o = 32; o > 0; o >>= 1) {
                        const unsigned long long y = __shfl_xor(key, o);
                        key = y < key ? y : key;
                    }
                    if (lane == tk) {
                        arg = key == ~0ull ? 0 : static_cast<int>(static_cast<uint32_t>(key));
                        best = key == ~0ull ? kFltMax : __uint_as_float(static_cast<uint32_t>(key >> 32));
                    }
                }
            }
        }
        if constexpr (EXACT != kLabelsOnly) {
            // the lane's own token row (in L2: its tiles were just read)
            km_u32x4_t xr[DP / 8];
            const uint16_t* src = kb + static_cast<int64_t>(min(t, a.T - 1)) * a.ts;
#pragma unroll
            for (int i = 0; i < DP / 8; ++i) xr[i] = *reinterpret_cast<const km_u32x4_t*>(src + 8 * i);
            auto dist = [&](int c) {
                return EXACT == kExactLds ? l2_lanes8_bf16<DP>(xr, cs + c * CS)
                                          : l2_lanes8_bf16<DP>(xr, cg + static_cast<int64_t>(c) * DP);
            };
            if (!every) {
                const int lo = pair ? min(c1, c2) : c1;
                const float d = dist(lo);
                if (d < best) {
                    best = d;
                    arg = lo;
                }
                if (pair) {
                    const int hi = max(c1, c2);
                    const float d2 = dist(hi);
                    if (d2 < best) {
                        best = d2;
                        arg = hi;
                    }
                }
            }
        }
        if (blk + 1 < blk1) {
            load_tokens(blk + 1);
        } else {   // (or the last block's would have to outlive the exhaustive form)
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int kh = 0; kh < KH; ++kh) bq[j][kh] = km_u32x4_t{0u, 0u, 0u, 0u};
        }
        if constexpr (EXACT == kLabelsOnly) {
            if (!every) arg = c1;
            // Tokens with two candidates, four at a time: lanes 16 i .. + 7
            // take the i-th token's lower candidate, + 8 .. + 15 the higher.
            // Lane part j sums dims j, j + 8, .. in ascending order (the
            // reference's lane j) and the first lane adds the eight sums left
            // to right (row shifts).
            uint64_t todo = __ballot(pair && valid);
            while (todo) {
                int s[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    s[i] = todo ? __builtin_ctzll(todo) : s[0];
                    todo &= todo - 1;
                }
                const int tk = grp == 0 ? s[0] : grp == 1 ? s[1] : grp == 2 ? s[2] : s[3];
                const int ca = __shfl(min(c1, c2), tk), cb = __shfl(max(c1, c2), tk);
                const int c = lane & 8 ? cb : ca;
                const int part = opaque(lane) & 7;
                const uint16_t* xrow = kb + static_cast<int64_t>(t0 + tk) * a.ts + part;
                const float* crow = cg + static_cast<int64_t>(c) * DP + part;
                uint16_t xv[DP / 8];
                float cv[DP / 8];
#pragma unroll
                for (int i = 0; i < DP / 8; ++i) {
                    xv[i] = xrow[8 * i];
                    cv[i] = crow[8 * i];
                }
                float acc = 0.0f;
#pragma unroll
                for (int i = 0; i < DP / 8; ++i) {
                    const float d = bf16_to_f32(xv[i]) - cv[i];
                    acc = __builtin_fmaf(d, d, acc);
                }
                float d = acc;
                d = d + dpp_row_shl<1>(acc);
                d = d + dpp_row_shl<2>(acc);
                d = d + dpp_row_shl<3>(acc);
                d = d + dpp_row_shl<4>(acc);
                d = d + dpp_row_shl<5>(acc);
                d = d + dpp_row_shl<6>(acc);
                d = d + dpp_row_shl<7>(acc);
                const float dh = dpp_row_shl<8>(d);   // the higher candidate's
                int win = d < kFltMax ? ca : 0;
                if (dh < (d < kFltMax ? d : kFltMax)) win = cb;
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int w = __builtin_amdgcn_readlane(win, 16 * i);
                    if (lane == s[i]) arg = w;
                }
            }
        }
        if (valid) {
            a.labels[static_cast<int64_t>(seg) * a.T + t] = arg;
            if (EXACT != kLabelsOnly && a.mind) a.mind[static_cast<int64_t>(seg) * a.T + t] = best;
        }
        if constexpr (EXACT != kLabelsOnly) {
            if (a.wpart) {   // inertia partial of the wave's 64 tokens
                const float part = wave_sum(valid ? best : 0.0f);
                if (lane == 0 && (t0 >> 6) < 4 * a.nblk) a.wpart[static_cast<int64_t>(seg) * 4 * a.nblk + (t0 >> 6)] = part;
            }
        }
    }
}

// ---------------------------------------------------------------- kmeans++
// kmeans_plusplus_init_inplace (kmeans_core.cpp:138-186) for every (head,
// subspace) segment at once, one launch per pick.  The random draws do not
// depend on the data: the host replays std::mt19937_64(seed) for the first
// index (uniform_int_distribution<int32_t>(0, T-1)) and for one
// generate_canonical<double, 53> per pick, which is what
// uniform_real_distribution<double>(0, total) consumes; target = canon *
// total.  The reference sums the min distances sequentially in double (the
// total, then the running sum that picks the first index with cumsum >=
// target).  When every value is a multiple of the smallest value's ulp and
// the total stays below 2^53 such units (the exponent spread is checked per
// pick), no partial sum rounds in double, whatever the order, so blocked
// sums equal the sequential ones; otherwise one thread replays the loops.
//
// Launch c >= 1 finds pick c - 1 (the first row, or from launch c - 1's block
// statistics and minima; every workgroup does, on its first wave, while its
// other loads are in flight), then updates each row's min distance to the
// picks and its block's statistics.  Minima and statistics alternate between
// two buffers, so launch c never overwrites what its own picks read.
//
//   km_pp_exact_kernel   the distance of every row: small inputs, which are
//                        bound by the chain of dependent loads of a pick (6.4
//                        us at 11k tokens, 8 segments; 13.1 us with the whole
//                        workgroup searching), and launch 1 of larger ones,
//                        which also makes an 8-bit copy of the rows
//   km_pp_screen_kernel  the later launches: only rows whose 8-bit copy
//                        cannot rule the new pick out get the distance
//   km_pp_pick_kernel    the last pick
//
// 8-bit copy: groups of 256 rows share one scale s_j per dim (largest
// magnitude / 127); x^ = s q.  With e >= |x - x^| over the group,
//   |x - c| >= |x^ - c| - e,
// so a row keeps its minimum m when |x^ - c| >= sqrt(m) + e.  |x^ - c|^2 =
// |x^|^2 + |c|^2 - 2 x^.c; x^.c = sum q_j (s_j c_j) runs on v_dot4_i32_i8
// against s_j c_j rounded to 16 bits (two 8-bit parts, exact integer sums, the
// rounding at most W / 2 per dim bounded apart).  fp32 rounding (at most 2^-17
// relative in the two norms, 2^-22 elsewhere, 2^-19 in the reference's
// distance) is covered by 2^-14 of the operands' magnitudes; NaN, infinities
// and norms past 1e37 get the distance.  What has no relative bound:
//   - a weight s_j c_j is rounded to a step W of at least kPpLeastWeight /
//     32512, so W / 2 holds for the smallest ones too and the quotient
//     32512 / (largest weight) stays finite;
//   - a product below the normal range (fp32 subnormals are kept) is off by at
//     most 2^-150: 2 * 128 * 127 of them in the dot product, 128 in each sum
//     of squares, together below 1e-40;
//   - an error e whose squares underflow is at most 5e-22 too small, and the
//     square root may take a subnormal minimum for zero (1.1e-19): beside
//     sqrt(m) + e <= 1e-9 their effect on the square, 2 (sqrt(m) + e) 5e-22
//     and 2 e 1.1e-19 + 1.2e-38, is below 1e-30 up to e = 4e-12 and below
//     2^-14 of the square beyond.
// The last two are the 1e-30 of the slack.
//
// The distance over some of the dims is a bound as well: each group's dims are
// copied in descending order of their scale, and a pick reads the first half
// of them (a quarter of the keys' bytes).  Only where a wave's rows that this
// half cannot rule out are more than half of them (keys without dominant
// channels, early picks) does it read the other half.  With the benchmark's
// keys (k = 64, 64 dims) 6 % of the rows change per pick, the whole copy
// leaves 7.8 % and its first half 9.8 %; k = 181: 2.5, 3.3 and 4.5 %.
constexpr int kPpScreenBytes = 16 << 20;   // key bytes from which the rows are copied to 8 bits
constexpr int64_t kPpCopyBytes = int64_t{4} << 30;   // largest copy
constexpr float kPpLeastWeight = 1e-30f;   // largest weight of a group that the steps of its 16 bits still follow

struct PpBlock {    // per (segment, block)
    double sum;     // of its min distances (exact when the exponent spread allows)
    int emin, emax; // exponent range of its non-zero values (emin = INT_MAX: none)
};

__device__ __forceinline__ int pp_exp(float m) {
    const int e = static_cast<int>((__float_as_uint(m) >> 23) & 0xFFu);
    return e > 0 ? e : 1;
}

// Exponent range of one non-negative value, into (emin, emax).
__device__ __forceinline__ void pp_range(float m, int& emin, int& emax) {
    if (m > 0.0f || m != m) {
        const int e = pp_exp(m);
        emin = min(emin, e);
        emax = max(emax, e);
    }
}

template <int CTRL, int ROW_MASK = 0xF>
__device__ __forceinline__ double dpp_f64(double v) {   // 0.0 where the source is outside
    const long long u = __double_as_longlong(v);
    const uint32_t lo = static_cast<uint32_t>(dpp_i<CTRL, ROW_MASK>(static_cast<int>(u)));
    const uint32_t hi = static_cast<uint32_t>(dpp_i<CTRL, ROW_MASK>(static_cast<int>(u >> 32)));
    return __longlong_as_double(static_cast<long long>((static_cast<unsigned long long>(hi) << 32) | lo));
}

// Inclusive prefix sum across the 64 lanes.
__device__ __forceinline__ double wave_incl_scan_f64(double v) {
    v += dpp_f64<0x111>(v);
    v += dpp_f64<0x112>(v);
    v += dpp_f64<0x114>(v);
    v += dpp_f64<0x118>(v);
    v += dpp_f64<0x142, 0xA>(v);
    v += dpp_f64<0x143, 0xC>(v);
    return v;
}

__device__ __forceinline__ double readlane_f64(double v, int lane) {
    const long long u = __double_as_longlong(v);
    const uint32_t lo = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(u), lane));
    const uint32_t hi = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(u >> 32), lane));
    return __longlong_as_double(static_cast<long long>((static_cast<unsigned long long>(hi) << 32) | lo));
}

// emin / emax over the wave (every lane): exponents are 1 .. 255.
__device__ __forceinline__ int wave_emin(int e) {
    const uint32_t inv = wave_max_u32(e == 0x7FFFFFFF ? 0u : 256u - static_cast<uint32_t>(e));
    return inv == 0 ? 0x7FFFFFFF : 256 - static_cast<int>(inv);
}
__device__ __forceinline__ int wave_emax(int e) { return static_cast<int>(wave_max_u32(static_cast<uint32_t>(e))); }

// First entry i (ascending) whose inclusive prefix base + v_0 + .. + v_i
// reaches target, over n entries held PER per lane (lane l: entries PER l ..);
// n - 1 if none does.  before: the exclusive prefix of that entry.
template <int PER>
__device__ __forceinline__ int pp_first_reaching(const double (&v)[PER], double base, double target, int n,
                                                 double& before) {
    double own = v[0];
#pragma unroll
    for (int u = 1; u < PER; ++u) own += v[u];
    const double incl = wave_incl_scan_f64(own) + base;
    const uint64_t hit = __ballot(incl >= target);
    const int l = hit ? __builtin_ctzll(hit) : 63;
    // every lane walks its own entries; lane l's walk is the answer
    double run = incl - own, at = run;
    int i = -1;
#pragma unroll
    for (int u = 0; u < PER; ++u) {
        if (i < 0 && run + v[u] >= target) {
            i = u;
            at = run;
        }
        run += v[u];
    }
    before = readlane_f64(at, l);
    const int u = __builtin_amdgcn_readlane(i, l);
    return hit && u >= 0 ? min(PER * l + u, n - 1) : n - 1;
}

// The reference's loops one addition after the other (the total, then the
// first row whose running sum reaches the target), by one wave: 64 rows per
// load, four loads ahead, each row added from its lane.  Both loops have the
// same running sums, so the second starts at the 64th part of the rows that
// the target lies in (their sums before are kept, one per lane).
// Bound by the chain of double additions: 23 ns per row, 3 ms per pick at
// 128k tokens, 16 segments (one lane with a load per addition: 20 ms; the same
// in a workgroup of 256 threads: 11 ms).
__device__ __forceinline__ int pp_sequential_row(const float* md, int T, double canon) {
    constexpr int AHEAD = 4, STEP = 16;
    const int lane = lane_id();
    const int part = (T + 4095) / 4096 * 64;   // rows per lane's part
    double sum = 0.0, before = 0.0, target = INFINITY;
    int first = 0, last = T;
    const auto load = [&](int i) { return i + lane < T ? md[i + lane] : 0.0f; };   // (a zero changes no sum)
#pragma unroll 1
    for (int pass = 0; pass < 2; ++pass) {
        float next[AHEAD];
#pragma unroll
        for (int u = 0; u < AHEAD; ++u) next[u] = load(first + 64 * u);
#pragma unroll 1
        for (int i = first; i < last; i += 64) {
            const float v = next[0];
#pragma unroll
            for (int u = 0; u + 1 < AHEAD; ++u) next[u] = next[u + 1];
            next[AHEAD - 1] = load(i + 64 * AHEAD);
            if (i % part == 0 && lane == i / part) before = sum;
            const auto row = [&](int j) {
                return static_cast<double>(__int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), j)));
            };
#pragma unroll 1
            for (int j0 = 0; j0 < 64; j0 += STEP) {
                double s = sum;
#pragma unroll
                for (int j = 0; j < STEP; ++j) sum += row(j0 + j);
                if (sum < target) continue;
#pragma unroll 1
                for (int j = 0; j < STEP; ++j) {
                    s += row(j0 + j);
                    if (s >= target) return i + j0 + j;
                }
            }
        }
        if (pass == 1) break;
        target = canon * sum + 0.0;
        // the last part that begins below the target (the first one otherwise)
        const int at = __popcll(__ballot(lane > 0 && lane * part < T && before < target));
        first = at * part;
        last = min(first + part, T);
        sum = at > 0 ? readlane_f64(before, at) : 0.0;
    }
    return 0;
}

// As a call, where the code in line made every pick longer (it is seldom
// run, but a pick is short: 6.24 against 6.55 us at 8k tokens, 6.8 against 7.0
// over 128 dims at 16k); with blocks of four groups the call's scratch would
// cost more (29.8 against 29.3 us at 128k).
__device__ __attribute__((noinline)) int pp_sequential_row_call(const float* md, int T, double canon) {
    return pp_sequential_row(md, T, canon);
}

// Row of pick c >= 1 of one segment (one wave; the row to every lane) from the
// minima md and block statistics st of the distance pass of pick c: blocks of
// 64 RPL rows.  kmeans_core.cpp:160-181.
template <int RPL>
__device__ int pp_pick_row(const float* md, const PpBlock* st, int nb, int T, double canon) {
    const int lane = lane_id();
    constexpr int SPER = 4;
    const int per = (nb + 63) / 64;
    int emin = 0x7FFFFFFF, emax = 0;
    double sums[SPER];
#pragma unroll
    for (int u = 0; u < SPER; ++u) sums[u] = 0.0;
    if (per <= SPER) {
        PpBlock e[SPER];
#pragma unroll
        for (int u = 0; u < SPER; ++u) e[u] = st[min(SPER * lane + u, nb - 1)];
#pragma unroll
        for (int u = 0; u < SPER; ++u)
            if (SPER * lane + u < nb) {
                sums[u] = e[u].sum;
                emin = min(emin, e[u].emin);
                emax = max(emax, e[u].emax);
            }
    } else {   // a run of `per` blocks per lane, searched again below
        const int b1 = min((lane + 1) * per, nb);
        for (int b = lane * per; b < b1; ++b) {
            const PpBlock e = st[b];
            sums[0] += e.sum;
            emin = min(emin, e.emin);
            emax = max(emax, e.emax);
        }
    }
    emin = wave_emin(emin);
    emax = wave_emax(emax);
    int logT = 0;
    while ((1ll << logT) < static_cast<long long>(T)) ++logT;
    if (__builtin_expect(emin != 0x7FFFFFFF && (emax - emin) + 24 + logT > 53, 0))
        return RPL == 16 ? pp_sequential_row(md, T, canon) : pp_sequential_row_call(md, T, canon);
    const double total = readlane_f64(wave_incl_scan_f64((sums[0] + sums[1]) + (sums[2] + sums[3])), 63);
    const double target = canon * total + 0.0;
    double base;
    int blk;
    if (per <= SPER) {
        blk = pp_first_reaching<SPER>(sums, 0.0, target, nb, base);
    } else {
        const double one[1] = {sums[0]};
        const int run = pp_first_reaching<1>(one, 0.0, target, 64, base);
        blk = min(run * per, nb - 1);
        for (int b0 = run * per; b0 < min((run + 1) * per, nb); b0 += 64) {   // one round up to 4096 blocks
            const double v[1] = {b0 + lane < min((run + 1) * per, nb) ? st[b0 + lane].sum : 0.0};
            const double all = readlane_f64(wave_incl_scan_f64(v[0]), 63);
            if (base + all >= target) {
                const double b = base;
                blk = b0 + pp_first_reaching<1>(v, b, target, 64, base);
                break;
            }
            base += all;
        }
    }
    // RPL consecutive rows per lane
    typedef float __attribute__((ext_vector_type(4), aligned(4))) f4;
    const int r0 = blk * 64 * RPL + lane * RPL;
    double v[RPL];
    if (r0 + RPL <= T) {
        f4 m[RPL / 4];
#pragma unroll
        for (int u = 0; u < RPL / 4; ++u) m[u] = *reinterpret_cast<const f4*>(md + r0 + 4 * u);
#pragma unroll
        for (int u = 0; u < RPL; ++u) v[u] = static_cast<double>(m[u / 4][u % 4]);
    } else {
#pragma unroll
        for (int u = 0; u < RPL; ++u) v[u] = r0 + u < T ? static_cast<double>(md[r0 + u]) : 0.0;
    }
    const int rows = min(64 * RPL, T - blk * 64 * RPL);
    return blk * 64 * RPL + pp_first_reaching<RPL>(v, base, target, rows, base);
}

typedef unsigned int __attribute__((ext_vector_type(4))) pp_u32x4_t;

struct PpStep {
    int c;                       // launch index: pick c - 1, distances to it
    int nbp;                     // blocks per segment
    int nsub;                    // blocks per workgroup
    int first[4];                // the first row, per subspace
    double canon[4];             // canon of pick c - 1 (c >= 2), per subspace
    const float* md_in;          // [seg][T] minima of launch c - 1
    float* md_out;               // [seg][T]
    const PpBlock* st_in;        // [seg][nbp] statistics of launch c - 1
    PpBlock* st_out;
    // the 8-bit copy by groups of 256 rows (RPT per block): [group][DP / 16][256]
    // rows' 16-byte chunks, their norms over the first half of the dims and
    // over all [group][2][256], the group's dims in the copy's order [group][DP]
    // and their scales, error bound [group]
    pp_u32x4_t* q;
    uint8_t* qd;
    float* qn;
    float* qs;
    float* qe;
};

// The new pick's row: found by the first wave, widened into cur (LDS) and, by
// the segment's first workgroup, written as a centroid.
template <int DP, int RPL>
__device__ __forceinline__ void pp_take_pick(const KmParams& a, const PpStep& ps, int seg, int p, const uint16_t* xb,
                                             float* cur) {
    if (threadIdx.x >= 64) return;
    const int lane = threadIdx.x, c = ps.c;
    const int sel = c == 1 ? ps.first[p]
                           : pp_pick_row<RPL>(ps.md_in + static_cast<int64_t>(seg) * a.T,
                                              ps.st_in + static_cast<int64_t>(seg) * ps.nbp, ps.nbp, a.T, ps.canon[p]);
    if (lane < DP / 8) {
        const pp_u32x4_t v = reinterpret_cast<const pp_u32x4_t*>(xb + static_cast<int64_t>(sel) * a.ts)[lane];
        const float4 f0 = make_float4(bf16_lo(v.x), bf16_hi(v.x), bf16_lo(v.y), bf16_hi(v.y));
        const float4 f1 = make_float4(bf16_lo(v.z), bf16_hi(v.z), bf16_lo(v.w), bf16_hi(v.w));
        reinterpret_cast<float4*>(cur)[2 * lane] = f0;
        reinterpret_cast<float4*>(cur)[2 * lane + 1] = f1;
        if (blockIdx.x == 0) {
            float4* dst = reinterpret_cast<float4*>(a.cent + (static_cast<int64_t>(seg) * a.kmax + c - 1) * DP);
            dst[2 * lane] = f0;
            dst[2 * lane + 1] = f1;
        }
    }
}

// Statistics of a block from its waves' (all 256 threads; one barrier).
__device__ __forceinline__ void pp_block_stats(double sum, int emin, int emax, PpBlock* sh, PpBlock* out) {
    const int w = threadIdx.x >> 6;
    const double s = readlane_f64(wave_incl_scan_f64(sum), 63);
    emin = wave_emin(emin);
    emax = wave_emax(emax);
    if (lane_id() == 0) sh[w] = PpBlock{s, emin, emax};
    __syncthreads();
    if (threadIdx.x == 0) {
        PpBlock o = sh[0];
        for (int i = 1; i < 4; ++i) {
            o.sum += sh[i].sum;
            o.emin = min(o.emin, sh[i].emin);
            o.emax = max(o.emax, sh[i].emax);
        }
        *out = o;
    }
}

// Rows are loaded coalesced (consecutive lanes read consecutive 16-byte
// chunks) and staged in LDS, from which each thread takes its own row.  RPT =
// 0: blocks of 256 rows; else launch 1 of the screened form, blocks of RPT
// such groups, whose 8-bit copy it writes.
template <int DP, int RPT>
__global__ __launch_bounds__(256) void km_pp_exact_kernel(KmParams a, PpStep ps) {
    constexpr bool FIRST = RPT > 0;
    __shared__ __attribute__((aligned(16))) float cur[DP];
    __shared__ PpBlock s_st[2][4];
    __shared__ float s_part[FIRST ? 512 : 1];
    __shared__ __attribute__((aligned(16))) float s_scale[FIRST ? DP : 4];
    __shared__ __attribute__((aligned(16))) float s_inv[FIRST ? DP : 4];
    __shared__ uint8_t s_dim[FIRST ? DP : 4];
    __shared__ float s_err[4];
    constexpr int CH = DP / 8;   // 16-byte chunks per row
    constexpr int GROUPS = FIRST ? RPT : 1;
    extern __shared__ __attribute__((aligned(16))) pp_u32x4_t s_rows[];   // [256][CH + 1]
    const int nb = ps.nbp, c = ps.c;
    const int seg = blockIdx.y, tid = threadIdx.x;
    const int h = seg / a.P, p = seg % a.P;
    if (c - 1 >= a.k[p]) return;
    const bool dist = c < a.k[p];   // false: pick c - 1 is the segment's last
    if (!dist && blockIdx.x != 0) return;
    const int T = a.T;
    const float* mdi = ps.md_in + static_cast<int64_t>(seg) * T;
    float* mdo = ps.md_out + static_cast<int64_t>(seg) * T;
    const uint16_t* xb = a.keys + static_cast<int64_t>(h) * a.hs + p * DP;
    const int blk0 = blockIdx.x * ps.nsub, blk1 = min(blk0 + ps.nsub, nb);
    // the first group does not depend on the pick: it is loaded before it
    pp_u32x4_t ld[CH];
    float prev = kFltMax;   // launch 1: no distances yet
    auto load_group = [&](int r0) {
        if (c > 1) prev = mdi[min(r0 + tid, T - 1)];
#pragma unroll
        for (int i = 0; i < CH; ++i) {
            const int f = tid + 256 * i;
            ld[i] = reinterpret_cast<const pp_u32x4_t*>(xb + static_cast<int64_t>(min(r0 + f / CH, T - 1)) * a.ts)[f % CH];
        }
    };
    if (dist) load_group(blk0 * 256 * GROUPS);
    pp_take_pick<DP, 4 * GROUPS>(a, ps, seg, p, xb, cur);
    if (!dist) return;
    for (int bk = blk0; bk < blk1; ++bk) {
        double sum = 0.0;
        int emin = 0x7FFFFFFF, emax = 0;
#pragma unroll 1
        for (int g = 0; g < GROUPS; ++g) {
            const int r0 = (bk * GROUPS + g) * 256;
            if (bk > blk0 || g > 0) {
                load_group(r0);
                __syncthreads();   // the previous group's rows are read
            }
#pragma unroll
            for (int i = 0; i < CH; ++i) {
                const int f = tid + 256 * i;
                s_rows[(f / CH) * (CH + 1) + f % CH] = ld[i];
            }
            __syncthreads();   // (and cur, before the first group)
            pp_u32x4_t v[CH];
#pragma unroll
            for (int i = 0; i < CH; ++i) v[i] = s_rows[tid * (CH + 1) + i];
            const int r = r0 + tid;
            const float d = l2_lanes8_bf16<DP>(v, cur);
            const float m = r < T ? (d < prev ? d : prev) : 0.0f;
            if (r < T) mdo[r] = m;
            sum += static_cast<double>(m);
            pp_range(m, emin, emax);
            if constexpr (FIRST) {
                // largest magnitude per dim: a dword column (two dims) per
                // thread over 256 / PARTS of the group's rows
                constexpr int COLS = DP / 2, PARTS = 256 / COLS;
                const uint32_t* words = reinterpret_cast<const uint32_t*>(s_rows);
                const int col = tid % COLS, part = tid / COLS;
                uint32_t lo = 0, hi = 0;   // |bf16| bits order like the values
                const int n = min(256, T - r0);
                for (int i = part * (256 / PARTS); i < (part + 1) * (256 / PARTS) && i < n; ++i) {
                    const uint32_t w = words[i * 4 * (CH + 1) + col] & 0x7FFF7FFFu;
                    lo = max(lo, w & 0xFFFFu);
                    hi = max(hi, w >> 16);
                }
                s_part[part * DP + 2 * col] = __uint_as_float(lo << 16);
                s_part[part * DP + 2 * col + 1] = __uint_as_float(hi << 16);
                __syncthreads();
                const int64_t group = (static_cast<int64_t>(seg) * nb + bk) * RPT + g;
                if (tid < DP) {
                    float m4 = 0.0f;   // (a NaN's bits give a NaN here, an infinity an infinite scale)
                    for (int i = 0; i < PARTS; ++i) m4 = s_part[i * DP + tid] > m4 || s_part[i * DP + tid] != s_part[i * DP + tid] ? s_part[i * DP + tid] : m4;
                    s_part[tid] = m4;   // (only this thread reads column tid of the parts)
                }
                __syncthreads();
                if (tid < DP) {
                    // place in descending order of magnitude (of its bits: a
                    // total order also over NaN), equal ones by dim
                    const uint32_t mine = __float_as_uint(s_part[tid]);
                    int at = 0;
#pragma unroll 8
                    for (int j = 0; j < DP; ++j) {
                        const uint32_t other = __float_as_uint(s_part[j]);
                        at += other > mine || (other == mine && j < tid) ? 1 : 0;
                    }
                    const float sc = s_part[tid] * (1.0f / 127.0f);
                    s_dim[at] = static_cast<uint8_t>(tid);
                    s_scale[at] = sc;
                    s_inv[at] = sc > 0.0f ? 1.0f / sc : 0.0f;
                    ps.qs[group * DP + at] = sc;
                    ps.qd[group * DP + at] = static_cast<uint8_t>(tid);
                }
                __syncthreads();
                const uint16_t* own = reinterpret_cast<const uint16_t*>(s_rows + tid * (CH + 1));
                float nrm = 0.0f, err = 0.0f;
#pragma unroll
                for (int i = 0; i < DP / 16; ++i) {
                    pp_u32x4_t o;
#pragma unroll
                    for (int w = 0; w < 4; ++w) {   // four dims per dword
                        uint32_t b = 0;
#pragma unroll
                        for (int e = 0; e < 4; ++e) {
                            const int j = 16 * i + 4 * w + e;
                            const float x = bf16_to_f32(own[s_dim[j]]);
                            const float t = fminf(fmaxf(rintf(x * s_inv[j]), -127.0f), 127.0f);
                            const float xh = t * s_scale[j];
                            nrm = __builtin_fmaf(xh, xh, nrm);
                            err = __builtin_fmaf(x - xh, x - xh, err);
                            b |= (static_cast<uint32_t>(static_cast<int>(t)) & 0xFFu) << (8 * e);
                        }
                        o[w] = b;
                    }
                    ps.q[(group * (DP / 16) + i) * 256 + tid] = o;
                    if (i == DP / 32 - 1) ps.qn[group * 512 + tid] = nrm;
                }
                ps.qn[group * 512 + 256 + tid] = nrm;
                // error bound of the group's rows; a non-finite one rules nothing out
                float e = r < T ? sqrtf(err) * (1.0f + 0x1p-14f) + 1e-30f : 0.0f;
                e = e <= 1e30f ? e : INFINITY;
                e = wave_max(e);
                if (lane_id() == 0) s_err[tid >> 6] = e;
                __syncthreads();
                if (tid == 0) ps.qe[group] = fmaxf(fmaxf(s_err[0], s_err[1]), fmaxf(s_err[2], s_err[3]));
            }
        }
        pp_block_stats(sum, emin, emax, s_st[(bk - blk0) & 1], ps.st_out + static_cast<int64_t>(seg) * nb + bk);
    }
}

// Launch c >= 2 of the screened form, over blocks of RPT groups of 256 rows.  A
// wave screens RPT rows per lane of one group (RPT = 4: group `wave` of the
// block; RPT = 1: a quarter of its only group, for inputs that would otherwise
// leave CUs idle): it weighs the group's scales with the pick, screens,
// queues the rows it cannot rule out and computes their distances 8 lanes per
// row (lane part j sums dims j, j + 8, .., the reference's lane j; row shifts
// add the eight sums left to right).  Only the block statistics cross waves.
//
// Bound by the copy's bytes (44 per 64-dim row with norm and minima, 80 when
// both halves are read) and the queue's dependent loads for large inputs, by
// the pick's dependent loads for small ones.  Per pick, 64 dims, 16 segments:
// 29.6 us at 128k tokens (22 us for the late picks; 33 us with the whole copy
// read, 55 us reading the keys), 106 us at 512k (146 and 250 us); keys without
// dominant channels read both halves one after the other, 7 % slower than the
// whole copy at once.  The next block's loads are issued before the queue (8
// lanes per row there: one row per lane spilled over 64 dims, 65 us).
template <int DP, int RPT>
__global__ __launch_bounds__(256, DP == 128 ? 2 : 4) void km_pp_screen_kernel(KmParams a, PpStep ps) {
    constexpr int CH = DP / 16;                   // 16-byte chunks per copied row
    constexpr int HC = CH / 2;                    // of the first half of the dims
    constexpr int DL = DP > 64 ? DP / 64 : 1;     // dims per lane of the weights
    __shared__ __attribute__((aligned(16))) float cur[DP];
    __shared__ PpBlock s_st[2][4];
    __shared__ __attribute__((aligned(16))) uint8_t s_w[4][2][DP];   // per wave: high and low weight bytes
    __shared__ uint16_t s_queue[4][64 * RPT];
    __shared__ float s_dist[4][64 * RPT];
    const int nb = ps.nbp, c = ps.c;
    const int seg = blockIdx.y, tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int h = seg / a.P, p = seg % a.P;
    if (c - 1 >= a.k[p]) return;
    const bool dist = c < a.k[p];
    if (!dist && blockIdx.x != 0) return;
    const int T = a.T;
    const float* mdi = ps.md_in + static_cast<int64_t>(seg) * T;
    float* mdo = ps.md_out + static_cast<int64_t>(seg) * T;
    const uint16_t* xb = a.keys + static_cast<int64_t>(h) * a.hs + p * DP;
    const int blk0 = blockIdx.x * ps.nsub, blk1 = min(blk0 + ps.nsub, nb);
    pp_u32x4_t q[RPT][HC];
    float m[RPT], nrm[RPT], sc[DL], err;
    int dim[DL];
    // the wave's group of block bk, its first row there and in the segment
    const int g_in = RPT == 4 ? wave : 0, row_in = RPT == 4 ? 0 : 64 * wave;
    static_assert(RPT == 4 || RPT == 1, "groups per block");
    auto group_of = [&](int bk) { return (static_cast<int64_t>(seg) * nb + bk) * RPT + g_in; };
    auto row_of = [&](int bk) { return (bk * RPT + g_in) * 256 + row_in; };
    auto load_group = [&](int bk) {
        const int64_t group = group_of(bk);
        const int r0 = row_of(bk);
#pragma unroll
        for (int u = 0; u < DL; ++u) {
            sc[u] = ps.qs[group * DP + (64 * u + lane) % DP];
            dim[u] = ps.qd[group * DP + (64 * u + lane) % DP];
        }
        err = ps.qe[group];
#pragma unroll
        for (int i = 0; i < RPT; ++i) {
            m[i] = mdi[min(r0 + 64 * i + lane, T - 1)];
            nrm[i] = ps.qn[group * 512 + row_in + 64 * i + lane];
#pragma unroll
            for (int k = 0; k < HC; ++k) q[i][k] = ps.q[(group * CH + k) * 256 + row_in + 64 * i + lane];
        }
    };
    if (dist) load_group(blk0);   // does not depend on the pick
    pp_take_pick<DP, 4 * RPT>(a, ps, seg, p, xb, cur);
    if (!dist) return;
    __syncthreads();
    float cp[DP / 8];   // dims part, part + 8, .. for the distances
#pragma unroll
    for (int i = 0; i < DP / 8; ++i) cp[i] = cur[8 * i + (lane & 7)];
#pragma unroll 1
    for (int bk = blk0; bk < blk1; ++bk) {
        const int64_t group = group_of(bk);
        const int r0 = row_of(bk);
        // 16-bit weights s_j c_j / W in two signed bytes; |c|^2 over the first
        // half of the dims and over all
        float wj[DL], wmax = 0.0f, cc1 = 0.0f, cc = 0.0f;
#pragma unroll
        for (int u = 0; u < DL; ++u) {
            const float cj = DP >= 64 || lane < DP ? cur[dim[u]] : 0.0f;
            wj[u] = sc[u] * cj;
            wmax = fmaxf(wmax, fabsf(wj[u]));
            if (64 * u + lane < DP / 2) cc1 = __builtin_fmaf(cj, cj, cc1);
            cc = __builtin_fmaf(cj, cj, cc);
        }
        wmax = wave_max(wmax);
        cc1 = wave_sum(cc1);
        // (weights below kPpLeastWeight are held at its steps: 32512 / wmax
        // would overflow from 9.6e-35 down, and a quotient of infinity makes
        // every weight, zero ones too, a largest one)
        const float wtop = fmaxf(wmax, kPpLeastWeight);
        const float W = wtop * (1.0f / 32512.0f), iw = 32512.0f / wtop;
#pragma unroll
        for (int u = 0; u < DL; ++u) {
            if (DP >= 64 || lane < DP) {
                const int t = static_cast<int>(fminf(fmaxf(rintf(wj[u] * iw), -32512.0f), 32512.0f));
                const int hi = (t + 128) >> 8;
                s_w[wave][0][64 * u + lane] = static_cast<uint8_t>(hi);
                s_w[wave][1][64 * u + lane] = static_cast<uint8_t>(t - 256 * hi);
            }
        }
        wave_lds_order();
        int hi[RPT], lo[RPT];
#pragma unroll
        for (int i = 0; i < RPT; ++i) hi[i] = lo[i] = 0;
        auto dot16 = [&](const pp_u32x4_t& x, int k, int i) {   // chunk k of row i
            const pp_u32x4_t wh = *reinterpret_cast<const pp_u32x4_t*>(&s_w[wave][0][16 * k]);
            const pp_u32x4_t wl = *reinterpret_cast<const pp_u32x4_t*>(&s_w[wave][1][16 * k]);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                hi[i] = __builtin_amdgcn_sdot4(static_cast<int>(x[e]), static_cast<int>(wh[e]), hi[i], false);
                lo[i] = __builtin_amdgcn_sdot4(static_cast<int>(x[e]), static_cast<int>(wl[e]), lo[i], false);
            }
        };
        // whether row i keeps its minimum: n = |x^|^2, c2 = |c|^2 over the dims
        // of the dot product.  The weights' rounding: at most W (1/2 + 2^-8) per
        // dim times |q| <= 127, twice.
        auto ruled_out = [&](int i, float n, float c2) {
            const float slack = 130.0f * DP * W + 0x1p-14f * c2 + 1e-30f;
            const float dot = W * static_cast<float>(256 * hi[i] + lo[i]);
            const float low = (n + c2) - 2.0f * dot - (slack + 0x1p-14f * n);
            const float reach = (__builtin_amdgcn_sqrtf(m[i]) + err) * (1.0f + 0x1p-14f);
            // (norms past 1e37 could overflow where the distance does not)
            return low >= reach * reach && n + c2 <= 1e37f;
        };
#pragma unroll
        for (int k = 0; k < HC; ++k)
#pragma unroll
            for (int i = 0; i < RPT; ++i) dot16(q[i][k], k, i);
        uint32_t need = 0;
        int left = 0;
#pragma unroll
        for (int i = 0; i < RPT; ++i) {
            const bool in = r0 + 64 * i + lane < T && m[i] != 0.0f && !ruled_out(i, nrm[i], cc1);
            if (in) need |= 1u << i;
            left += __popcll(__ballot(in));
        }
        // a row's distance costs four times what its other half does
        if (left > 32 * RPT) {
            const float c2 = wave_sum(cc);
            float all[RPT];
#pragma unroll
            for (int i = 0; i < RPT; ++i) {
                all[i] = ps.qn[group * 512 + 256 + row_in + 64 * i + lane];
#pragma unroll
                for (int k = 0; k < HC; ++k) q[i][k] = ps.q[(group * CH + HC + k) * 256 + row_in + 64 * i + lane];
            }
#pragma unroll
            for (int k = 0; k < HC; ++k)
#pragma unroll
                for (int i = 0; i < RPT; ++i) dot16(q[i][k], HC + k, i);
#pragma unroll
            for (int i = 0; i < RPT; ++i)
                if (ruled_out(i, all[i], c2)) need &= ~(1u << i);
        }
        // the next block's loads overlap with the queue's
        float mc[RPT];
#pragma unroll
        for (int i = 0; i < RPT; ++i) mc[i] = m[i];
        if (bk + 1 < blk1) load_group(bk + 1);
        // the queue: this wave's rows in (i, lane) order
        int nq = 0;
#pragma unroll
        for (int i = 0; i < RPT; ++i) {
            const bool in = (need >> i) & 1u;
            const uint64_t bal = __ballot(in);
            if (in) s_queue[wave][nq + __popcll(bal & lanemask_lt())] = static_cast<uint16_t>(64 * i + lane);
            nq += __popcll(bal);
        }
        wave_lds_order();
#pragma unroll 1
        for (int e0 = 0; e0 < nq; e0 += 16) {   // 16 rows, two per 8 lanes
            int id[2];
            uint16_t xv[2][DP / 8];
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                id[u] = s_queue[wave][min(e0 + 8 * u + (lane >> 3), nq - 1)];
                const uint16_t* row = xb + static_cast<int64_t>(r0 + id[u]) * a.ts + (lane & 7);
#pragma unroll
                for (int i = 0; i < DP / 8; ++i) xv[u][i] = row[8 * i];
            }
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                float acc = 0.0f;
#pragma unroll
                for (int i = 0; i < DP / 8; ++i) {
                    const float d = bf16_to_f32(xv[u][i]) - cp[i];
                    acc = __builtin_fmaf(d, d, acc);
                }
                float d = acc;
                d = d + dpp_row_shl<1>(acc);
                d = d + dpp_row_shl<2>(acc);
                d = d + dpp_row_shl<3>(acc);
                d = d + dpp_row_shl<4>(acc);
                d = d + dpp_row_shl<5>(acc);
                d = d + dpp_row_shl<6>(acc);
                d = d + dpp_row_shl<7>(acc);
                if ((lane & 7) == 0) s_dist[wave][id[u]] = d;
            }
        }
        wave_lds_order();
        double sum = 0.0;
        int emin = 0x7FFFFFFF, emax = 0;
#pragma unroll
        for (int i = 0; i < RPT; ++i) {
            const int r = r0 + 64 * i + lane;
            float v = mc[i];
            if ((need >> i) & 1u) {
                const float d = s_dist[wave][64 * i + lane];
                if (d < v) v = d;
            }
            if (r < T) {
                mdo[r] = v;
                sum += static_cast<double>(v);
                pp_range(v, emin, emax);
            }
        }
        pp_block_stats(sum, emin, emax, s_st[(bk - blk0) & 1], ps.st_out + static_cast<int64_t>(seg) * nb + bk);
    }
}

// The last pick c of every segment with k == c + 1 (c == 0: the first row)
// from the minima and statistics of launch c (blocks of 64 RPL rows).
template <int DP, int RPL>
__global__ __launch_bounds__(64) void km_pp_pick_kernel(KmParams a, PpStep ps) {
    const int seg = blockIdx.x, lane = threadIdx.x;
    const int h = seg / a.P, p = seg % a.P;
    const int c = ps.c;
    if (c >= a.k[p]) return;
    const uint16_t* xb = a.keys + static_cast<int64_t>(h) * a.hs + p * DP;
    const int sel = c == 0 ? ps.first[p]
                           : pp_pick_row<RPL>(ps.md_in + static_cast<int64_t>(seg) * a.T,
                                              ps.st_in + static_cast<int64_t>(seg) * ps.nbp, ps.nbp, a.T, ps.canon[p]);
    float* dst = a.cent + (static_cast<int64_t>(seg) * a.kmax + c) * DP;
    for (int d = lane; d < DP; d += 64) dst[d] = bf16_to_f32(xb[static_cast<int64_t>(sel) * a.ts + d]);
}

// Early stop (kmeans_core.cpp:244-262) of one segment.  The inertia has a fixed
// reduction order: the four wave partials of each 256-token block, contiguous
// blocks per thread, lanes, then waves.  prev alternates between two slots,
// so that several workgroups can run the test of one iteration.
__device__ __forceinline__ float stop_block_partial(const KmParams& a, int seg, int b) {
    const float* wp = a.wpart + static_cast<int64_t>(seg) * 4 * a.nblk;
    const int nw = (a.T + 63) / 64;   // wave partials written
    float v[4];
#pragma unroll
    for (int w = 0; w < 4; ++w) v[w] = 4 * b + w < nw ? wp[4 * b + w] : 0.0f;
    return ((v[0] + v[1]) + v[2]) + v[3];
}

__device__ __forceinline__ bool stop_test(const KmParams& a, int seg, int it, float inertia, bool record) {
    const float prev = a.prev[2 * seg + (it & 1)];
    const float change = fabsf(prev - inertia);
    const float rel = prev > 0.0f ? change / prev : 0.0f;
    const bool min_ok = (it + 1) >= (a.es_min > 1 ? a.es_min : 1);
    const bool stop = min_ok && (rel <= fmaxf(0.0f, a.es_rel) || change <= fmaxf(0.0f, a.tol));
    if (record) {
        if (a.iters) a.iters[seg] = it + 1;
        if (stop)
            a.done[seg] = 1;
        else
            a.prev[2 * seg + ((it + 1) & 1)] = inertia;
    }
    return stop;
}

__global__ __launch_bounds__(1024) void km_stop_kernel(KmParams a, int it) {
    __shared__ float sred[16];
    const int seg = blockIdx.x, tid = threadIdx.x;
    if (a.done[seg]) return;
    const int per = (a.nblk + 1023) / 1024;
    float part = 0.0f;
    for (int b = tid * per; b < (tid + 1) * per && b < a.nblk; ++b) part += stop_block_partial(a, seg, b);
    part = wave_sum(part);
    if ((tid & 63) == 0) sred[tid >> 6] = part;
    __syncthreads();
    if (tid == 0) {
        float inertia = 0.0f;
        for (int w = 0; w < 16; ++w) inertia += sred[w];
        stop_test(a, seg, it, inertia, true);
    }
}

// Member lists by superblocks of a.sbt tokens: each workgroup puts its
// tokens in label order (ascending token inside a label) into its own slice
// of `sorted` and writes the superblock's row of label offsets (loff[0 .. k]:
// first place of each label, then the token count).  The ordered slice goes
// through LDS (coalesced stores) up to kStagedItems tokens.  11.6 us at 128k
// tokens, 16 segments; superblocks of thousands of tokens keep the M-step's
// member search and its column of label offsets short (58 us per M-step; 62
// against 68 us with one row of offsets per 256 tokens in an earlier form), and serve any T (a scan over
// per-block histograms and a scatter took 340 us at 512k tokens, k = 181; this
// kernel 34 us).
__host__ __device__ inline size_t members_lds_bytes(int waves, int kmax, int sbt) {
    return (static_cast<size_t>(waves) * kmax + 32) * sizeof(int) + (sbt <= kStagedItems ? 2 * static_cast<size_t>(sbt) : 0);
}

__global__ __launch_bounds__(1024) void km_members_kernel(KmParams a) {
    extern __shared__ int smem_i[];
    const int seg = blockIdx.y, sb = blockIdx.x;
    if (a.done && a.done[seg]) return;
    const int k = a.k[seg % a.P];
    int* cnt = smem_i;                                          // [waves][k]
    int* wsum = smem_i + (blockDim.x >> 6) * a.kmax;            // [16]
    uint16_t* staged = reinterpret_cast<uint16_t*>(wsum + 32);  // [sbt]
    const bool stage = a.sbt <= kStagedItems;
    const int base = sb * a.sbt;
    const int m = min(a.sbt, a.T - base);
    const int32_t* lab = a.labels + static_cast<int64_t>(seg) * a.T + base;
    int32_t* out = a.sorted + static_cast<int64_t>(seg) * a.T + base;
    int32_t* row = a.loff + (static_cast<int64_t>(seg) * a.nsb + sb) * (a.kmax + 1);
    if (threadIdx.x == 0) row[k] = m;
    superblock_sort(
        m, a.sbt, k, cnt, wsum, [&](int i) { return lab[i]; }, [&](int c, int first) { row[c] = first; },
        [&](int i, int at) {
            if (stage)
                staged[at] = static_cast<uint16_t>(i);
            else
                out[at] = base + i;
        });
    if (!stage) return;
    __syncthreads();
    for (int i = threadIdx.x; i < m; i += blockDim.x) out[i] = base + staged[i];
}

// Empty clusters whose ordinal falls in [e0, e0 + kMoreDraws): the draws of
// that slice (clusters beyond kDraws empty ones only occur when k > kDraws).
// A thread per cluster (256 of them from 256 blk on) looks, its wave copies
// the rows of those that it finds (seldom any).  768 draws are 3 KB of kernel
// arguments: one launch up to k = 1024 (8 x 1018 clusters: 4.6 us per
// iteration; three launches of 256 draws with a workgroup per cluster 14 us).
constexpr int kMoreDraws = 768;
struct MoreDraws {
    int32_t v[kMoreDraws];
};

__device__ __forceinline__ void reseed(const KmParams& a, const MoreDraws& draws, int e0, int blk, int seg) {
    const int c = blk * 256 + threadIdx.x;
    const int h = seg / a.P, p = seg % a.P, lane = lane_id();
    const int e = c < a.k[p] ? a.empties[static_cast<int64_t>(seg) * a.kmax + c] - e0 : -1;
    for (uint64_t hit = __ballot(e >= 0 && e < kMoreDraws); hit; hit &= hit - 1) {
        const int l = __builtin_ctzll(hit);
        const int tok = draws.v[__builtin_amdgcn_readlane(e, l)];
        const uint16_t* row = a.keys + h * a.hs + p * a.DP + static_cast<int64_t>(tok) * a.ts;
        float* dst = a.cent + (static_cast<int64_t>(seg) * a.kmax + (c - lane + l)) * a.DP;
        for (int d = lane; d < a.DP; d += 64) dst[d] = bf16_to_f32(row[d]);
    }
}

__global__ __launch_bounds__(256) void km_reseed_kernel(KmParams a, MoreDraws draws, int e0) {
    const int seg = blockIdx.y;
    if (a.done && a.done[seg]) return;
    reseed(a, draws, e0, blockIdx.x, seg);
}

// Members up to which one wave sums a cluster (km_update_wave_kernel); of a
// larger one it leaves -1 minus its size in `empties`.
constexpr int kWaveMost = 512;

// The n-th of those clusters of a segment, or -1 (every wave looks).
__device__ __forceinline__ int nth_large(const KmParams& a, int seg, int n) {
    const int k = a.k[seg % a.P], lane = lane_id();
    const int32_t* size = a.empties + static_cast<int64_t>(seg) * a.kmax;
    for (int c0 = 0; c0 < k; c0 += 256) {
        int v[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) v[u] = size[min(c0 + 64 * u + lane, k - 1)];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            uint64_t hit = __ballot(v[u] < -1 && c0 + 64 * u + lane < k);
            if (n < __popcll(hit)) {
                for (; n > 0; --n) hit &= hit - 1;
                return c0 + 64 * u + __builtin_ctzll(hit);
            }
            n -= __popcll(hit);
        }
    }
    return -1;
}

// M-step, one workgroup per cluster: wave 0 keeps the chains (lane d =
// dimension d, members in ascending token order, one dependent fp32 add
// each) while waves 1..3 gather the member rows, so a large cluster streams
// with three waves' worth of loads in flight.  Batch b (64 rows) belongs to
// loader 1 + b % 3 as its local batch b / 3; round q hands batches 3q ..
// 3q+2 over through one of two sets of LDS slots (the loaders fill round
// q+1 while wave 0 sums round q), one barrier per round.  Each loader keeps
// NB local batches in flight in a register ring and loads the member ids 2 NB
// local batches ahead.
// SUPER: a power of two, at least the superblocks (the member search's steps).
// SUPER = 0: no member lists; every workgroup scans the segment's labels
// itself (a quarter per wave, the matching tokens to the wave's LDS slice, in
// order), and runs the early-stop test of the iteration.  For the shortest
// contexts the two launches this saves cost more than the scan: at 11k
// tokens, k = 32, 4 heads, 11.8 us against 8.3 + 4.8 us (and 3.1 us for a stop
// test) plus the launches between.
// Draw = MoreDraws: what km_update_wave_kernel leaves, the n-th cluster of
// more than kWaveMost members for workgroup n of the first a.T / (kWaveMost +
// 1), and behind them the empty clusters past its draws (it: their first
// ordinal).
template <int DP, int SUPER, typename Draw>
__global__ __launch_bounds__(256) void km_update_block_kernel(KmParams a, Draw draws, int it) {
    constexpr bool SCAN = SUPER == 0;
    constexpr bool REST = std::is_same<Draw, MoreDraws>::value;
    constexpr int PARTS = DP / 8;    // 16-byte parts per row
    constexpr int RPL = 64 / PARTS;  // rows per load instruction
    constexpr int LPB = PARTS;       // load instructions per 64-row batch
    constexpr int NL = 3;            // loader waves
    // local batches in flight per loader (register ring).  Two: every
    // workgroup fills its ring at the start, and with four the burst (~75 MB
    // at configs[1]) delayed the first rounds of the largest clusters, whose
    // chains set the kernel's length (79.9 -> 71.4 us per M-step).
    constexpr int NB = 2;
    constexpr int HALVES = DP > 64 ? DP / 64 : 1;   // dims per chain lane
    __shared__ km_u32x4_t ring[2 * NL][64 * PARTS];
    // the label's exclusive prefix over the superblocks, its first place in
    // each, the waves' member counts
    __shared__ int s_pref[SCAN ? 1 : kMaxSuper];
    __shared__ int s_lof[SCAN ? 1 : kMaxSuper];
    __shared__ int s_wt[4];
    __shared__ int s_emp;
    __shared__ int s_stop;
    __shared__ uint8_t s_seen[SCAN ? kImiMaxK : 1];
    extern __shared__ uint16_t s_list[];   // SCAN: [4][span]
    const int seg = blockIdx.y;
    const int h = seg / a.P, p = seg % a.P;
    if (a.done && a.done[seg]) return;
    int c = blockIdx.x;
    if constexpr (REST) {
        const int large = gridDim.x - (a.kmax + 255) / 256;
        if (c >= large) {
            reseed(a, draws, it, c - large, seg);
            return;
        }
        c = nth_large(a, seg, c);
        if (c < 0) return;
    }
    if (c >= a.k[p]) return;
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const uint16_t* kbase = a.keys + h * a.hs + p * DP;
    float* dst = a.cent + (static_cast<int64_t>(seg) * a.kmax + c) * DP;
    const int32_t* rows = a.loff + static_cast<int64_t>(seg) * a.nsb * (a.kmax + 1);
    const int32_t* lab = a.labels + static_cast<int64_t>(seg) * a.T;
    const int span = (a.T + 255) / 256 * 64;   // SCAN: tokens per wave
    if (tid == 0) s_emp = 0;
    if constexpr (SCAN) {
        if (a.exact && wave == 0) {   // at most 64 blocks: one per lane
            const float inertia = wave_sum(lane < a.nblk ? stop_block_partial(a, seg, lane) : 0.0f);
            const bool stop = stop_test(a, seg, it, inertia, c == 0 && lane == 0);
            if (lane == 0) s_stop = stop;
        }
        const int w0 = wave * span, w1 = min(w0 + span, a.T);
        int run = 0;
        // four consecutive labels per lane and load, eight loads in flight
        typedef int __attribute__((ext_vector_type(4), aligned(4))) i32x4;
        for (int i = w0; i < w1; i += 2048) {
            i32x4 l[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                const int tk = i + 256 * u + 4 * lane;
                if (tk + 4 <= a.T) {
                    l[u] = *reinterpret_cast<const i32x4*>(lab + tk);
                } else {
#pragma unroll
                    for (int e = 0; e < 4; ++e) l[u][e] = tk + e < a.T ? lab[tk + e] : -1;
                }
            }
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                if (i + 256 * u >= w1) break;
                const int tk = i + 256 * u + 4 * lane;
                bool hit[4];
                int cnt = 0;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    hit[e] = l[u][e] == c && tk + e < w1;
                    cnt += hit[e];
                }
                const int incl = wave_incl_scan(cnt);
                int at = w0 + run + incl - cnt;
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (hit[e]) s_list[at++] = static_cast<uint16_t>(tk + e);
                run += __builtin_amdgcn_readlane(incl, 63);
            }
        }
        if (lane == 0) s_wt[wave] = run;
        __syncthreads();
        if (a.exact && s_stop) return;
    } else {
        // this label's first place and count in every superblock (two per
        // thread, their offset pairs loaded together), then the prefix of the
        // counts
        int cv[kMaxSuper / 256], lv[kMaxSuper / 256];
#pragma unroll
        for (int u = 0; u < kMaxSuper / 256; ++u) {
            const int32_t* r = rows + static_cast<int64_t>(min(2 * tid + u, a.nsb - 1)) * (a.kmax + 1) + c;
            lv[u] = r[0];
            cv[u] = r[1];
        }
#pragma unroll
        for (int u = 0; u < kMaxSuper / 256; ++u) cv[u] = 2 * tid + u < a.nsb ? cv[u] - lv[u] : 0;
        const int both = cv[0] + cv[1];
        const int incl = wave_incl_scan(both);
        if (lane == 63) s_wt[wave] = incl;
        __syncthreads();
        int before = incl - both;
        for (int w = 0; w < wave; ++w) before += s_wt[w];
        if (2 * tid < a.nsb) {
            s_pref[2 * tid] = before;
            s_lof[2 * tid] = lv[0];
        }
        if (2 * tid + 1 < a.nsb) {
            s_pref[2 * tid + 1] = before + cv[0];
            s_lof[2 * tid + 1] = lv[1];
        }
        __syncthreads();
    }
    const int n = (s_wt[0] + s_wt[1]) + (s_wt[2] + s_wt[3]);
    if (!REST && n == 0) {
        // the empty ordinal: labels below c with no member
        if constexpr (SCAN) {
            for (int c2 = tid; c2 < c; c2 += 256) s_seen[c2] = 0;
            __syncthreads();
            for (int i = tid; i < a.T; i += 256) s_seen[lab[i]] = 1;
            __syncthreads();
        }
        for (int c2 = tid; c2 < c; c2 += 256) {
            int any = SCAN ? s_seen[c2] : 0;
            if (!SCAN)
            for (int b = 0; b < a.nsb; ++b) {
                const int32_t* r = rows + static_cast<int64_t>(b) * (a.kmax + 1) + c2;
                any |= r[1] - r[0];
            }
            if (any == 0) atomicAdd(&s_emp, 1);
        }
        __syncthreads();
        const int e = s_emp;
        if (tid == 0) a.empties[static_cast<int64_t>(seg) * a.kmax + c] = e;   // past this launch's draws: km_reseed_kernel
        if (wave == 0 && e < kDraws) {
            const int tok = draws.v[e];
            for (int d = lane; d < DP; d += 64) dst[d] = bf16_to_f32(kbase[static_cast<int64_t>(tok) * a.ts + d]);
        }
        return;
    }
    if (!REST && tid == 0) a.empties[static_cast<int64_t>(seg) * a.kmax + c] = -1;
    const int nb = (n + 63) >> 6;              // 64-row batches
    const int rounds = (nb + NL - 1) / NL;     // = local batches of loader 1
    const int32_t* lst = a.sorted + static_cast<int64_t>(seg) * a.T;
    // member j: the superblock holding it (the last one whose prefix is <= j)
    // and its place there
    const int p1 = s_wt[0], p2 = p1 + s_wt[1], p3 = p2 + s_wt[2];
    auto member = [&](int j) {
        if constexpr (SCAN)
            return static_cast<int>(s_list[j < p1 ? j : j < p2 ? span + j - p1 : j < p3 ? 2 * span + j - p2 : 3 * span + j - p3]);
        int b = 0;
#pragma unroll
        for (int step = SUPER / 2; step > 0; step >>= 1)
            b = (b + step < a.nsb && s_pref[b + step] <= j) ? b + step : b;
        return lst[static_cast<int64_t>(b) * a.sbt + s_lof[b] + (j - s_pref[b])];
    };
    // rounds padded to whole ring cycles: the loaders' loop body is then free
    // of branches, so the compiler's wait before each slot write counts the
    // loads issued since that batch's (a branch around a load makes it assume
    // the fewest, which waited for nearly every load and left one batch in
    // flight).  Padding rounds re-read the last member's row (L2-resident)
    // and are not summed.
    const int rounds_pad = (rounds + NB - 1) / NB * NB;
    if (wave > 0) {
        const int lw = wave - 1;
        const int part = lane % PARTS, rsub = lane / PARTS;
        // member ids of local batch q (global batch NL q + lw); past n the
        // last member again (a valid row, never summed: the chain adds only
        // the first n).  No select on the loaded id: one would make the
        // compiler wait for each id load right after issuing it.
#define KMB_ID(q) member(min((NL * (q) + lw) * 64 + lane, n - 1))
#define KMB_ROWS(idv, slot)                                                                            \
    _Pragma("unroll") for (int u = 0; u < LPB; ++u) {                                                \
        const int id_ = __shfl((idv), u * RPL + rsub);                                               \
        rr[slot][u] = *reinterpret_cast<const km_u32x4_t*>(kbase + static_cast<int64_t>(id_) * a.ts + part * 8); \
    }
        // rows of local batches 0 .. NB-1 in the register ring, ids of
        // NB .. 2NB-1 in the id ring; round q writes batch q, loads the rows
        // of q + NB and the ids of q + 2NB
        // (the prologue issues its loads in the loop's order -- slot j's rows,
        // then slot j's next ids -- so the waits inside the loop are the same
        // on entry and on the back edge)
        int idr[NB], id0[NB];
        km_u32x4_t rr[NB][LPB];
#pragma unroll
        for (int j = 0; j < NB; ++j) id0[j] = KMB_ID(j);
#pragma unroll
        for (int j = 0; j < NB; ++j) {
            KMB_ROWS(id0[j], j)
            idr[j] = KMB_ID(NB + j);
            __builtin_amdgcn_sched_barrier(0);   // keep this order (no reordering of the loads)
        }
#pragma unroll 1
        for (int q0 = 0; q0 < rounds_pad; q0 += NB) {
#pragma unroll
            for (int j = 0; j < NB; ++j) {
                const int q = q0 + j;
                km_u32x4_t* slot = ring[(q & 1) * NL + lw];
#pragma unroll
                for (int u = 0; u < LPB; ++u) slot[(u * RPL + rsub) * PARTS + part] = rr[j][u];
                KMB_ROWS(idr[j], j)
                idr[j] = KMB_ID(q + 2 * NB);
                __syncthreads();
            }
        }
#undef KMB_ID
#undef KMB_ROWS
    } else {
        float acc[HALVES];
#pragma unroll
        for (int hh = 0; hh < HALVES; ++hh) acc[hh] = 0.0f;
#pragma unroll 1
        for (int q = 0; q < rounds_pad; ++q) {
            __syncthreads();   // round q's slots are filled
            if (q >= rounds) continue;
            if (HALVES == 1 && NL * 64 * (q + 1) <= n) {
                // a full round (three batches of 64 members): the next batch's
                // reads are issued before the current batch's additions, and
                // the widening of value j + 1 is scheduled between the adds of
                // j - 1 and j, so no add waits on the instruction before it
                const int lg = lane >> 4, ln = lane & 15;
                const int boff = (ln >> 2) * DP + 16 * (lg % (DP / 16)) + 4 * (ln & 3);
                km_u32x2_t w[2][16];
#pragma unroll
                for (int i = 0; i < 16; ++i)
                    w[0][i] = __builtin_bit_cast(
                        km_u32x2_t,
                        __builtin_amdgcn_ds_read_tr16_b64_v4i16((km_lds_s16x4_t*)(reinterpret_cast<const uint16_t*>(
                                                                    ring[(q & 1) * NL]) + boff + 4 * i * DP)));
#pragma unroll
                for (int lw = 0; lw < NL; ++lw) {
                    if (lw + 1 < NL) {
#pragma unroll
                        for (int i = 0; i < 16; ++i)
                            w[(lw + 1) & 1][i] = __builtin_bit_cast(
                                km_u32x2_t, __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                                                (km_lds_s16x4_t*)(reinterpret_cast<const uint16_t*>(
                                                                      ring[(q & 1) * NL + lw + 1]) + boff + 4 * i * DP)));
                    }
                    float f[64];
#pragma unroll
                    for (int i = 0; i < 16; ++i) {
                        f[4 * i] = __uint_as_float(w[lw & 1][i][0] << 16);
                        f[4 * i + 1] = __uint_as_float(w[lw & 1][i][0] & 0xFFFF0000u);
                        f[4 * i + 2] = __uint_as_float(w[lw & 1][i][1] << 16);
                        f[4 * i + 3] = __uint_as_float(w[lw & 1][i][1] & 0xFFFF0000u);
                    }
#pragma unroll
                    for (int j = 0; j < 64; ++j) acc[0] = acc[0] + f[j];
                }
                continue;
            }
#pragma unroll
            for (int lw = 0; lw < NL; ++lw) {
                const int b = NL * q + lw;
                if (b < nb) {
                    const uint16_t* rows = reinterpret_cast<const uint16_t*>(ring[(q & 1) * NL + lw]);
                    const int cnt = (n - 64 * b) < 64 ? (n - 64 * b) : 64;
                    if (cnt == 64) {
                        // transposing reads: 16-lane group g takes the 4 x 16
                        // block of members 4i..4i+3, dims 16 (g % (DP/16)) ..
                        // +15, so lane d holds dim d of four consecutive
                        // members per read (lanes >= DP read a copy and are
                        // not stored); all 16 reads in flight at once.  DP =
                        // 128: a second pass over dims 64..127.
                        const int lg = lane >> 4, ln = lane & 15;
#pragma unroll
                        for (int hh = 0; hh < HALVES; ++hh) {
                            const uint16_t* base =
                                rows + (ln >> 2) * DP + 64 * hh + 16 * (lg % (DP / 16)) + 4 * (ln & 3);
                            km_u32x2_t w[16];
#pragma unroll
                            for (int i = 0; i < 16; ++i)
                                w[i] = __builtin_bit_cast(
                                    km_u32x2_t, __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                                                    (km_lds_s16x4_t*)(base + 4 * i * DP)));
#pragma unroll
                            for (int i = 0; i < 16; ++i) {
                                acc[hh] = acc[hh] + __uint_as_float(w[i][0] << 16);
                                acc[hh] = acc[hh] + __uint_as_float(w[i][0] & 0xFFFF0000u);
                                acc[hh] = acc[hh] + __uint_as_float(w[i][1] << 16);
                                acc[hh] = acc[hh] + __uint_as_float(w[i][1] & 0xFFFF0000u);
                            }
                        }
                    } else {
#pragma unroll
                        for (int hh = 0; hh < HALVES; ++hh)
                            if (64 * hh + lane < DP)
                                for (int r = 0; r < cnt; ++r)
                                    acc[hh] = acc[hh] + bf16_to_f32(rows[r * DP + 64 * hh + lane]);
                    }
                }
            }
        }
#pragma unroll
        for (int hh = 0; hh < HALVES; ++hh)
            if (64 * hh + lane < DP) dst[64 * hh + lane] = acc[hh] * (1.0f / static_cast<float>(n));
    }
}

// M-step of small clusters over 128 dims (IVF: about 16 members each): one wave
// per cluster, lane l the chains of dims 2l and 2l + 1, kWaveRows member rows
// (one dword per lane) in flight.  A workgroup per cluster spends its time on
// the hand-off between its waves: 120 us per M-step for 8 x 1018 clusters of
// 16 members, 17 us here.  Bound by its loads' latency, 65 ns per member, so a
// cluster of more than kWaveMost members goes to a workgroup of the launch
// that follows anyway for the re-seeding (12 ns per member): with 8k of 16k
// keys in one cluster an M-step takes 0.12 ms, 0.5 when its wave summed it.
constexpr int kWaveRows = 32;
constexpr int kWaveClusters = 4;
constexpr int kWaveMaxMean = 64;   // mean members per cluster up to which it is used

template <int SUPER>
__global__ __launch_bounds__(64 * kWaveClusters) void km_update_wave_kernel(KmParams a, Draws draws) {
    __shared__ int s_pref[kWaveClusters][SUPER];
    __shared__ int s_lof[kWaveClusters][SUPER];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int c = blockIdx.x * kWaveClusters + wave, seg = blockIdx.y;
    const int h = seg / a.P, p = seg % a.P;
    if (c >= a.k[p]) return;   // (no barrier below: a wave works alone)
    if (a.done && a.done[seg]) return;
    const uint16_t* kbase = a.keys + h * a.hs + p * 128;
    float* dst = a.cent + (static_cast<int64_t>(seg) * a.kmax + c) * 128;
    const int32_t* rows = a.loff + static_cast<int64_t>(seg) * a.nsb * (a.kmax + 1);
    int n = 0;
    for (int b0 = 0; b0 < a.nsb; b0 += 64) {
        const int b = b0 + lane;
        const int32_t* r = rows + static_cast<int64_t>(min(b, a.nsb - 1)) * (a.kmax + 1) + c;
        const int lof = r[0], cnt = b < a.nsb ? r[1] - lof : 0;
        const int incl = wave_incl_scan(cnt);
        if (b < a.nsb) {
            s_pref[wave][b] = n + incl - cnt;
            s_lof[wave][b] = lof;
        }
        n += __builtin_amdgcn_readlane(incl, 63);
    }
    wave_lds_order();
    int32_t* empty = a.empties + static_cast<int64_t>(seg) * a.kmax + c;
    if (n == 0) {
        int e = 0;   // empty labels below c
        for (int c2 = lane; c2 < c; c2 += 64) {
            int any = 0;
            for (int b = 0; b < a.nsb; ++b) {
                const int32_t* r = rows + static_cast<int64_t>(b) * (a.kmax + 1) + c2;
                any |= r[1] - r[0];
            }
            e += any == 0 ? 1 : 0;
        }
        e = wave_sum_i(e);
        if (lane == 0) *empty = e;   // past this launch's draws: km_reseed_kernel
        if (e < kDraws) {
            const uint32_t v =
                reinterpret_cast<const uint32_t*>(kbase + static_cast<int64_t>(draws.v[e]) * a.ts)[lane];
            *reinterpret_cast<float2*>(dst + 2 * lane) = make_float2(bf16_lo(v), bf16_hi(v));
        }
        return;
    }
    if (lane == 0) *empty = n > kWaveMost ? -1 - n : -1;
    if (n > kWaveMost) return;
    const int32_t* lst = a.sorted + static_cast<int64_t>(seg) * a.T;
    auto member = [&](int j) {   // as in km_update_block_kernel
        int b = 0;
#pragma unroll
        for (int step = SUPER / 2; step > 0; step >>= 1)
            b = (b + step < a.nsb && s_pref[wave][b + step] <= j) ? b + step : b;
        return lst[static_cast<int64_t>(b) * a.sbt + s_lof[wave][b] + (j - s_pref[wave][b])];
    };
    float x0 = 0.0f, x1 = 0.0f;
    int id = member(min(lane, n - 1));
    for (int j0 = 0; j0 < n; j0 += 64) {
        const int nid = member(min(j0 + 64 + lane, n - 1));
#pragma unroll 1
        for (int half = 0; half < 64; half += kWaveRows) {
            if (j0 + half >= n) break;
            // rows past the last member re-read it and are not added
            uint32_t v[kWaveRows];
#pragma unroll
            for (int u = 0; u < kWaveRows; ++u) {
                const int t = __builtin_amdgcn_readlane(id, half + u);
                v[u] = reinterpret_cast<const uint32_t*>(kbase + static_cast<int64_t>(t) * a.ts)[lane];
            }
#pragma unroll
            for (int u = 0; u < kWaveRows; ++u)
                if (j0 + half + u < n) {
                    x0 = x0 + bf16_lo(v[u]);
                    x1 = x1 + bf16_hi(v[u]);
                }
        }
        id = nid;
    }
    const float inv = 1.0f / static_cast<float>(n);
    *reinterpret_cast<float2*>(dst + 2 * lane) = make_float2(x0 * inv, x1 * inv);
}

__global__ void km_reset_kernel(KmParams a) {
    const int seg = blockIdx.x * blockDim.x + threadIdx.x;
    if (seg >= a.H * a.P) return;
    a.prev[2 * seg] = a.prev[2 * seg + 1] = 3.402823466e38f;
    if (a.done) a.done[seg] = 0;
    if (a.iters) a.iters[seg] = a.done ? 0 : a.max_iters;   // km_stop counts them with early stop
}

int validate(const imi_kmeans_args* a, int& kmax, int& dp) {
    IMI_REQUIRE(a != nullptr, IMI_ERR_INVALID, "imi_kmeans: null args");
    IMI_REQUIRE(a->keys && a->centroids && a->labels, IMI_ERR_INVALID, "imi_kmeans: null pointer argument");
    IMI_REQUIRE(a->kv_heads > 0 && a->n_tokens > 0, IMI_ERR_INVALID, "imi_kmeans: empty input (H=%d T=%d)",
                a->kv_heads, a->n_tokens);
    IMI_REQUIRE(a->parts == 1 || a->parts == 2 || a->parts == 4, IMI_ERR_UNSUPPORTED,
                "imi_kmeans: parts must be 1 (IVF), 2 or 4 (got %d)", a->parts);
    IMI_REQUIRE(a->dim % a->parts == 0, IMI_ERR_INVALID, "imi_kmeans: dim %d not divisible by parts %d", a->dim,
                a->parts);
    dp = a->dim / a->parts;
    IMI_REQUIRE(dp == 32 || dp == 64 || (a->parts == 1 && dp == 128), IMI_ERR_UNSUPPORTED,
                "imi_kmeans: subspace width %d unsupported (32 or 64; 128 for IVF)", dp);
    IMI_REQUIRE(a->max_iters >= 1, IMI_ERR_INVALID, "imi_kmeans: max_iters must be >= 1");
    const int kcap = a->parts == 1 ? kIvfMaxK : kImiMaxK;
    kmax = 0;
    for (int p = 0; p < a->parts; ++p) {
        IMI_REQUIRE(a->k[p] >= 1 && a->k[p] <= kcap, IMI_ERR_UNSUPPORTED, "imi_kmeans: k[%d]=%d outside [1,%d]", p,
                    a->k[p], kcap);
        kmax = a->k[p] > kmax ? a->k[p] : kmax;
    }
    IMI_REQUIRE(a->init_mode >= 0 && a->init_mode <= 2, IMI_ERR_INVALID,
                "imi_kmeans: init_mode %d (0 first-k, 1 given, 2 kmeans++)", a->init_mode);
    if (a->init_mode == 0)
        IMI_REQUIRE(kmax <= a->n_tokens, IMI_ERR_INVALID,
                    "imi_kmeans: first-k initialisation needs n_tokens (%d) >= k (%d)", a->n_tokens, kmax);
    IMI_REQUIRE((a->token_stride % 8) == 0 && (a->head_stride % 8) == 0, IMI_ERR_INVALID,
                "imi_kmeans: strides must be multiples of 8 elements (16-byte rows)");
    IMI_REQUIRE((reinterpret_cast<uintptr_t>(a->keys) & 15) == 0, IMI_ERR_INVALID,
                "imi_kmeans: keys must be 16-byte aligned");
    return IMI_OK;
}

// Whether kmeans++ screens its rows over an 8-bit copy: from 16 MB of keys
// (below, a pick is bound by its dependent loads and the copy would not pay;
// 8k tokens, 16 segments) while the copy stays below 4 GB.
bool pp_screened(int T, int segs, int dp) {
    const int64_t elems = static_cast<int64_t>(T) * segs * dp;
    return 2 * elems >= kPpScreenBytes && elems <= kPpCopyBytes;
}

// Groups of 256 rows per block of the screened passes: four, but one while
// blocks of four would be fewer than kPpFewBlocks (two workgroups per CU): 8
// heads of 16k tokens over 128 dims (128 blocks of four) take 7.1 us per pick
// with one group, 9.1 us with four and 17.5 us reading the keys; 40k tokens
// over 64 dims, 16 segments (640 blocks) 16.2, 15.1 and 22 us.
constexpr int kPpFewBlocks = 512;
int pp_groups(int T, int segs) {
    return static_cast<int64_t>((T + 1023) / 1024) * segs >= kPpFewBlocks ? 4 : 1;
}

template <int DP, int RPT>
int run_plusplus(const KmParams& p, const imi_kmeans_args* a, int segs, hipStream_t stream) {
    // kmeans++ seeds 42, 43, 44, 45 by subspace, the same for every head
    // (kmeans_core.cpp:459, 469; IVF: seed 42, kmeans_core.cpp:548-556)
    PpStep ps{};
    std::vector<double> canon[4];
    for (int part = 0; part < a->parts; ++part) {
        std::mt19937_64 rng(static_cast<uint64_t>(42 + part));
        std::uniform_int_distribution<int32_t> first(0, a->n_tokens - 1);
        ps.first[part] = first(rng);
        canon[part].assign(a->k[part], 0.0);
        for (int c = 1; c < a->k[part]; ++c)
            canon[part][c] = std::generate_canonical<double, std::numeric_limits<double>::digits>(rng);
    }
    constexpr bool screened = RPT > 0;
    const int rows = screened ? 256 * RPT : 256;
    const int nbp = (p.T + rows - 1) / rows;
    ps.nbp = nbp;
    ps.q = reinterpret_cast<pp_u32x4_t*>(p.ppq);
    ps.qd = p.ppqd;
    ps.qn = p.ppqn;
    ps.qs = p.ppqs;
    ps.qe = p.ppqe;
    PpBlock* st = static_cast<PpBlock*>(p.ppstats);
    // minima and statistics alternate between two buffers (one of them the
    // member lists' `sorted`, free until the first M-step)
    float* md[2] = {p.ppmd, reinterpret_cast<float*>(p.sorted)};
    PpBlock* sts[2] = {st, st + static_cast<size_t>(segs) * nbp};
    const size_t lds = static_cast<size_t>(256) * (DP / 8 + 1) * 16;
    // one resident round of workgroups, each over nsub consecutive blocks
    const auto sub_blocks = [&](const void* fn, size_t dyn) {
        int per_cu = 0;
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, fn, 256, dyn) != hipSuccess || per_cu <= 0) per_cu = 1;
        const int64_t want = static_cast<int64_t>(per_cu) * device_cus();
        return static_cast<int>(std::max<int64_t>(1, (static_cast<int64_t>(nbp) * segs + want - 1) / want));
    };
    const void* exact_fn = reinterpret_cast<const void*>(&km_pp_exact_kernel<DP, RPT>);
    if (DP == 128)   // 68 KB of LDS per workgroup
        IMI_HIP_CHECK(hipFuncSetAttribute(exact_fn, hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(lds)));
    const int sub_first = sub_blocks(exact_fn, lds);
    int sub_next = sub_first;
    if constexpr (screened) sub_next = sub_blocks(reinterpret_cast<const void*>(&km_pp_screen_kernel<DP, RPT>), 0);
    // launch c (1 <= c < kmax): pick c - 1 and the distances to it
    for (int c = 1; c < p.kmax; ++c) {
        ps.c = c;
        for (int part = 0; part < a->parts; ++part)
            ps.canon[part] = c - 1 >= 1 && c - 1 < a->k[part] ? canon[part][c - 1] : 0.0;
        ps.md_in = md[(c - 1) & 1];
        ps.md_out = md[c & 1];
        ps.st_in = sts[(c - 1) & 1];
        ps.st_out = sts[c & 1];
        ps.nsub = c == 1 ? sub_first : sub_next;
        const dim3 grid((nbp + ps.nsub - 1) / ps.nsub, segs);
        if (!screened || c == 1)
            hipLaunchKernelGGL((km_pp_exact_kernel<DP, RPT>), grid, dim3(256), lds, stream, p, ps);
        else if constexpr (screened)
            hipLaunchKernelGGL((km_pp_screen_kernel<DP, RPT>), grid, dim3(256), 0, stream, p, ps);
        IMI_LAUNCH_CHECK("kmeans++ pass");
    }
    // the last pick of the segments with kmax centroids
    const int c = p.kmax - 1;
    ps.c = c;
    for (int part = 0; part < a->parts; ++part) ps.canon[part] = c >= 1 && c < a->k[part] ? canon[part][c] : 0.0;
    ps.md_in = md[c & 1];
    ps.st_in = sts[c & 1];
    ps.md_out = nullptr;
    ps.st_out = nullptr;
    hipLaunchKernelGGL((km_pp_pick_kernel<DP, screened ? 4 * RPT : 4>), dim3(segs), dim3(64), 0, stream, p, ps);
    IMI_LAUNCH_CHECK("km_pp_pick_kernel");
    return IMI_OK;
}

template <int DP>
int seed_plusplus(const KmParams& p, const imi_kmeans_args* a, int segs, int groups, hipStream_t stream) {
    return groups == 4   ? run_plusplus<DP, 4>(p, a, segs, stream)
           : groups == 1 ? run_plusplus<DP, 1>(p, a, segs, stream)
                         : run_plusplus<DP, 0>(p, a, segs, stream);
}

// Whether a run's kmeans++ would screen its rows.
bool seeds_screened(const imi_kmeans_args* a) {
    return a->init_mode == 2 && pp_screened(a->n_tokens, a->kv_heads * a->parts, a->dim / a->parts);
}

// screened: with the 8-bit copy of a screened kmeans++ (seeds_screened).
size_t workspace_bytes(const imi_kmeans_args* a, int kmax, bool screened, KmParams* out) {
    const int segs = a->kv_heads * a->parts;
    const int nblk = (a->n_tokens + 255) / 256;
    Carver cv(a->workspace);
    KmParams p{};
    superblocks(a->n_tokens, segs, p.sbt, p.nsb);
    p.wpart = cv.take<float>(static_cast<size_t>(segs) * 4 * nblk);
    p.sorted = cv.take<int32_t>(static_cast<size_t>(segs) * a->n_tokens);
    p.loff = cv.take<int32_t>(static_cast<size_t>(segs) * p.nsb * (kmax + 1));
    p.empties = cv.take<int32_t>(static_cast<size_t>(segs) * kmax);
    p.prev = cv.take<float>(2 * segs);
    p.done = cv.take<int32_t>(segs);
    if (a->init_mode == 2) {
        const int dp = a->dim / a->parts;
        const size_t rows = 256 * (screened ? pp_groups(a->n_tokens, segs) : 1);   // per block
        const size_t blocks = (a->n_tokens + rows - 1) / rows * segs;
        p.ppstats = cv.take<PpBlock>(2 * blocks);   // two launches' worth
        p.ppmd = cv.take<float>(static_cast<size_t>(segs) * a->n_tokens);
        if (screened) {
            p.ppq = cv.take<uint8_t>(blocks * rows * dp);
            p.ppqd = cv.take<uint8_t>(blocks * rows / 256 * dp);
            p.ppqn = cv.take<float>(2 * blocks * rows);
            p.ppqs = cv.take<float>(blocks * rows / 256 * dp);
            p.ppqe = cv.take<float>(blocks * rows / 256);
        }
    }
    if (out) *out = p;
    return cv.used();
}

template <int DP, int NW, bool STREAM, int EXACT>
int launch_screen(const KmParams& p, int segs, size_t lds, hipStream_t stream) {
    const void* fn = reinterpret_cast<const void*>(&km_screen_kernel<DP, NW, STREAM, EXACT>);
    if (lds > 64 * 1024)
        IMI_HIP_CHECK(hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(lds)));
    // as many workgroups as fit on the device at once, each over `chunks`
    // consecutive blocks of 64 NW tokens
    int per_cu = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, km_screen_kernel<DP, NW, STREAM, EXACT>, 64 * NW, lds) !=
            hipSuccess ||
        per_cu <= 0)
        per_cu = 1;
    const int nblk = (p.T + 64 * NW - 1) / (64 * NW);
    // or one fewer per CU, where the CU with the most blocks then has at least
    // 1/16 fewer of them (4-way at 64k tokens, 8 heads: 5 workgroups of 7 blocks
    // on some CUs and 4 on others took 16 % longer than 4 of 8 on each)
    int chunks = 1;
    int64_t most = 0;
    for (int w = per_cu; w >= std::max(1, per_cu - 1); --w) {
        const int64_t want = static_cast<int64_t>(w) * device_cus();
        const int64_t c = std::max<int64_t>(1, (static_cast<int64_t>(nblk) * segs + want - 1) / want);
        const int64_t groups = (nblk + c - 1) / c * segs;
        const int64_t blocks = (groups + device_cus() - 1) / device_cus() * c;
        if (most == 0 || 16 * blocks <= 15 * most) {
            chunks = static_cast<int>(c);
            most = blocks;
        }
    }
    hipLaunchKernelGGL((km_screen_kernel<DP, NW, STREAM, EXACT>), dim3((nblk + chunks - 1) / chunks, segs),
                       dim3(64 * NW), lds, stream, p, chunks);
    IMI_LAUNCH_CHECK("km_screen_kernel");
    return IMI_OK;
}

// p.exact: the distances are read (min distances or the early-stop inertia);
// their fp32 centroid rows stay in LDS beside the packed tiles up to 150 KB.
// Four waves per workgroup while at least two workgroups' centroids fit in a
// CU's LDS, eight beyond.
template <int DP>
int run_assign(const KmParams& p, int segs, hipStream_t stream) {
    using L = ScreenLds<DP>;
    if constexpr (DP == 128) {
        const size_t lds = L::packed(2 * kChunkTiles);
        return p.exact ? launch_screen<DP, 4, true, kExactGlobal>(p, segs, lds, stream)
                       : launch_screen<DP, 4, true, kLabelsOnly>(p, segs, lds, stream);
    } else {
        const size_t lds = L::packed((p.kmax + 15) / 16);
        if (!p.exact)
            return lds <= 52 * 1024 ? launch_screen<DP, 4, false, kLabelsOnly>(p, segs, lds, stream)
                                    : launch_screen<DP, 8, false, kLabelsOnly>(p, segs, lds, stream);
        const size_t both = lds + L::rows(p.kmax);
        if (both <= 150 * 1024)
            return both <= 52 * 1024 ? launch_screen<DP, 4, false, kExactLds>(p, segs, both, stream)
                                     : launch_screen<DP, 8, false, kExactLds>(p, segs, both, stream);
        return launch_screen<DP, 8, false, kExactGlobal>(p, segs, lds, stream);
    }
}

// Whether the M-step scans the labels itself (km_update_block_kernel, SUPER =
// 0): up to 16384 tokens (16-bit list entries, at most 64 blocks for the stop
// test) and 2^19 (token, cluster) pairs per segment, so that the workgroups of
// a segment read at most 2 MB of labels from L2.
bool scans_labels(const KmParams& p) {
    return p.DP <= 64 && p.T <= 16384 && static_cast<int64_t>(p.T) * p.kmax <= (1 << 19);
}

// Whether one wave sums a cluster (km_update_wave_kernel; the large ones are
// left to the launches of run_rest).
bool sums_by_wave(const KmParams& p) {
    return p.DP == 128 && p.T <= static_cast<int64_t>(kWaveMaxMean) * p.kmax;
}

template <int DP>
int run_update(const KmParams& p, int segs, const Draws& dr, int it, hipStream_t stream) {
    if (sums_by_wave(p)) {
        const dim3 grid((p.kmax + kWaveClusters - 1) / kWaveClusters, segs);
        if (p.nsb <= 32)
            hipLaunchKernelGGL(km_update_wave_kernel<32>, grid, dim3(64 * kWaveClusters), 0, stream, p, dr);
        else
            hipLaunchKernelGGL(km_update_wave_kernel<kMaxSuper>, grid, dim3(64 * kWaveClusters), 0, stream, p, dr);
        IMI_LAUNCH_CHECK("km_update_wave_kernel");
        return IMI_OK;
    }
    const dim3 grid(p.kmax, segs);
    if (DP <= 64 && scans_labels(p)) {
        constexpr int W = DP <= 64 ? DP : 64;
        const size_t lists = static_cast<size_t>((p.T + 255) / 256) * 512;   // beside the ring and its like
        IMI_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(&km_update_block_kernel<W, 0, Draws>),
                                          hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(lists)));
        hipLaunchKernelGGL((km_update_block_kernel<W, 0, Draws>), grid, dim3(256), lists, stream, p, dr, it);
    } else if (p.nsb <= 32)
        hipLaunchKernelGGL((km_update_block_kernel<DP, 32, Draws>), grid, dim3(256), 0, stream, p, dr, it);
    else
        hipLaunchKernelGGL((km_update_block_kernel<DP, kMaxSuper, Draws>), grid, dim3(256), 0, stream, p, dr, it);
    IMI_LAUNCH_CHECK("km_update_block_kernel");
    return IMI_OK;
}

// After run_update: the clusters too large for one wave, and the draws of
// empty ordinals kDraws and up (`draw` continues the iteration's sequence).
template <typename Next>
int run_rest(const KmParams& p, int segs, Next draw, hipStream_t stream) {
    int large = sums_by_wave(p) ? p.T / (kWaveMost + 1) : 0;
    for (int e0 = kDraws; e0 < p.kmax || large > 0; e0 += kMoreDraws) {
        MoreDraws more;
        for (int e = e0; e < std::min(p.kmax, e0 + kMoreDraws); ++e) more.v[e - e0] = draw();
        const dim3 grid(large + (p.kmax + 255) / 256, segs);
        if (large == 0)
            hipLaunchKernelGGL(km_reseed_kernel, grid, dim3(256), 0, stream, p, more, e0);
        else if (p.nsb <= 32)
            hipLaunchKernelGGL((km_update_block_kernel<128, 32, MoreDraws>), grid, dim3(256), 0, stream, p, more, e0);
        else
            hipLaunchKernelGGL((km_update_block_kernel<128, kMaxSuper, MoreDraws>), grid, dim3(256), 0, stream, p, more, e0);
        IMI_LAUNCH_CHECK("the launch after the M-step");
        large = 0;
    }
    return IMI_OK;
}

int run_members(const KmParams& p, int segs, hipStream_t stream) {
    const int waves = sort_waves(p.kmax);
    const size_t lds = members_lds_bytes(waves, p.kmax, p.sbt);
    if (lds > 64 * 1024)
        IMI_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(&km_members_kernel),
                                          hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(lds)));
    hipLaunchKernelGGL(km_members_kernel, dim3(p.nsb, segs), dim3(64 * waves), lds, stream, p);
    IMI_LAUNCH_CHECK("km_members_kernel");
    return IMI_OK;
}

}  // namespace
}  // namespace imi

using namespace imi;

static int kmeans_workspace_size(const imi_kmeans_args* a, size_t* bytes, bool least) {
    clear_error();
    int kmax, dp;
    int rc = validate(a, kmax, dp);
    if (rc) return rc;
    IMI_REQUIRE(bytes != nullptr, IMI_ERR_INVALID, "imi_kmeans_workspace_size: null output");
    imi_kmeans_args tmp = *a;
    tmp.workspace = nullptr;
    *bytes = workspace_bytes(&tmp, kmax, !least && seeds_screened(a), nullptr);
    return IMI_OK;
}

extern "C" int imi_kmeans_workspace_size(const imi_kmeans_args* a, size_t* bytes) {
    return kmeans_workspace_size(a, bytes, false);
}

extern "C" int imi_kmeans_min_workspace_size(const imi_kmeans_args* a, size_t* bytes) {
    return kmeans_workspace_size(a, bytes, true);
}

extern "C" int imi_kmeans_execute(const imi_kmeans_args* a, imi_stream_t stream_) {
    clear_error();
    hipStream_t stream = reinterpret_cast<hipStream_t>(stream_);
    int kmax, dp;
    int rc = validate(a, kmax, dp);
    if (rc) return rc;
    imi_kmeans_args tmp = *a;
    tmp.workspace = nullptr;
    const size_t need = workspace_bytes(&tmp, kmax, false, nullptr);
    IMI_REQUIRE(a->workspace != nullptr && a->workspace_bytes >= need, IMI_ERR_WORKSPACE,
                "imi_kmeans_execute: workspace %zu bytes < %zu required", a->workspace_bytes, need);
    const bool screened = seeds_screened(a) && a->workspace_bytes >= workspace_bytes(&tmp, kmax, true, nullptr);

    KmParams p;
    workspace_bytes(a, kmax, screened, &p);
    p.keys = a->keys;
    p.hs = a->head_stride;
    p.ts = a->token_stride;
    p.H = a->kv_heads;
    p.T = a->n_tokens;
    p.P = a->parts;
    p.kmax = kmax;
    p.DP = dp;
    for (int i = 0; i < 4; ++i) p.k[i] = i < a->parts ? a->k[i] : 0;
    p.cent = a->centroids;
    p.labels = a->labels;
    p.mind = nullptr;
    p.iters = a->iters_run;
    p.nblk = (a->n_tokens + 255) / 256;
    p.max_iters = a->max_iters;
    p.tol = a->tol;
    p.es_min = a->early_stop_min_iter;
    p.es_rel = a->early_stop_rel_tol;
    const int segs = a->kv_heads * a->parts;
    const bool early_stop = a->early_stop_min_iter <= a->max_iters;
    if (!early_stop) p.done = nullptr;  // no test can fire: skip the flag reads

    hipLaunchKernelGGL(km_reset_kernel, dim3((segs + 63) / 64), dim3(64), 0, stream, p);
    IMI_LAUNCH_CHECK("km_reset_kernel");
    if (a->init_mode == 0) {
        hipLaunchKernelGGL(km_init_first_kernel, dim3(kmax, segs), dim3(64), 0, stream, p);
        IMI_LAUNCH_CHECK("km_init_first_kernel");
    } else if (a->init_mode == 2) {
        const int groups = screened ? pp_groups(a->n_tokens, segs) : 0;
        rc = dp == 128 ? seed_plusplus<128>(p, a, segs, groups, stream)
                       : (dp == 64 ? seed_plusplus<64>(p, a, segs, groups, stream)
                                   : seed_plusplus<32>(p, a, segs, groups, stream));
        if (rc) return rc;
    }
    for (int it = 0; it < a->max_iters; ++it) {
        // the inertia of iteration it enters the stop tests of it and it + 1
        p.exact = early_stop && it + 2 >= std::max(a->early_stop_min_iter, 1) ? 1 : 0;
        rc = dp == 128 ? run_assign<128>(p, segs, stream)
                       : (dp == 64 ? run_assign<64>(p, segs, stream) : run_assign<32>(p, segs, stream));
        if (rc) return rc;
        if (!scans_labels(p)) {
            if (p.exact) {   // (before, no test can fire)
                hipLaunchKernelGGL(km_stop_kernel, dim3(segs), dim3(1024), 0, stream, p, it);
                IMI_LAUNCH_CHECK("km_stop_kernel");
            }
            rc = run_members(p, segs, stream);
            if (rc) return rc;
        }
        // Empty-cluster draws of this iteration: std::mt19937(it + 12345) with
        // uniform_int_distribution<int32_t>(0, T-1), one per empty cluster in
        // ascending cluster order (kmeans_core.cpp:299-311).
        Draws dr;
        std::mt19937 rng(static_cast<unsigned>(it + 12345));
        std::uniform_int_distribution<int32_t> dist(0, a->n_tokens - 1);
        for (int e = 0; e < std::min(kmax, kDraws); ++e) dr.v[e] = dist(rng);
        rc = dp == 128 ? run_update<128>(p, segs, dr, it, stream)
                       : (dp == 64 ? run_update<64>(p, segs, dr, it, stream) : run_update<32>(p, segs, dr, it, stream));
        if (rc) return rc;
        rc = run_rest(p, segs, [&] { return dist(rng); }, stream);
        if (rc) return rc;
    }
    return IMI_OK;
}

extern "C" int imi_kmeans_assign(const uint16_t* keys, int64_t head_stride, int64_t token_stride, int32_t kv_heads,
                                 int32_t n_tokens, int32_t dim, int32_t parts, const int32_t* k,
                                 const float* centroids, int32_t* labels, float* mind, imi_stream_t stream_) {
    clear_error();
    imi_kmeans_args a{};
    a.keys = keys;
    a.head_stride = head_stride;
    a.token_stride = token_stride;
    a.kv_heads = kv_heads;
    a.n_tokens = n_tokens;
    a.dim = dim;
    a.parts = parts;
    IMI_REQUIRE(k != nullptr, IMI_ERR_INVALID, "imi_kmeans_assign: null k");
    for (int i = 0; i < parts && i < 4; ++i) a.k[i] = k[i];
    a.max_iters = 1;
    a.init_mode = 1;
    a.centroids = const_cast<float*>(centroids);
    a.labels = labels;
    int kmax, dp;
    int rc = validate(&a, kmax, dp);
    if (rc) return rc;
    KmParams p{};
    p.keys = keys;
    p.hs = head_stride;
    p.ts = token_stride;
    p.H = kv_heads;
    p.T = n_tokens;
    p.P = parts;
    p.kmax = kmax;
    p.DP = dp;
    for (int i = 0; i < 4; ++i) p.k[i] = i < parts ? k[i] : 0;
    p.cent = const_cast<float*>(centroids);
    p.labels = labels;
    p.mind = mind;
    p.exact = mind != nullptr ? 1 : 0;
    p.nblk = (n_tokens + 255) / 256;
    hipStream_t stream = reinterpret_cast<hipStream_t>(stream_);
    if (dp == 128) return run_assign<128>(p, kv_heads * parts, stream);
    return dp == 64 ? run_assign<64>(p, kv_heads * parts, stream) : run_assign<32>(p, kv_heads * parts, stream);
}
