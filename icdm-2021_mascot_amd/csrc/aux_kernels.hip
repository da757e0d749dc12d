// Kernels around the update loop: binary16 <-> binary32 conversion, grouped-storage scatter and
// gather, the g-switching error estimate, test RMSE (dense and grouped), model init, histogram,
// re-indexing.  All are streaming, HBM-bound, grid-stride kernels.
#include "mf_host.h"
#include "mf_device.h"
#include <type_traits>
#include <cmath>
#include <vector>

namespace mf {

constexpr int kStreamBlock = 256;
static inline uint32_t stream_grid(uint64_t n, int per_thread = 1)
{
    uint64_t blocks = (n + (uint64_t)kStreamBlock * per_thread - 1) / ((uint64_t)kStreamBlock * per_thread);
    const uint64_t cap = 256ull * 32;             // 32 workgroups per CU keeps every XCD busy
    if (blocks > cap) blocks = cap;
    if (blocks == 0) blocks = 1;
    return (uint32_t)blocks;
}

// ---- conversions (model_init.cu:85-112, precision_switching.h:1-6) -----------------------------
__global__ __launch_bounds__(kStreamBlock) void float2half_kernel(const float* __restrict__ in, uint16_t* __restrict__ out, uint64_t n)
{
    const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    const uint64_t n2 = n / 2;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n2; i += stride) {
        const float2 v = reinterpret_cast<const float2*>(in)[i];
        half2_t h; h.x = (half_t)v.x; h.y = (half_t)v.y;
        reinterpret_cast<uint32_t*>(out)[i] = bits(h);
    }
    if ((n & 1) && blockIdx.x == 0 && threadIdx.x == 0) out[n - 1] = (uint16_t)bits((half_t)in[n - 1]);
}
__global__ __launch_bounds__(kStreamBlock) void half2float_kernel(const uint16_t* __restrict__ in, float* __restrict__ out, uint64_t n)
{
    const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    const uint64_t n2 = n / 2;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n2; i += stride) {
        const half2_t h = from_bits<half2_t>(reinterpret_cast<const uint32_t*>(in)[i]);
        reinterpret_cast<float2*>(out)[i] = make_float2((float)h.x, (float)h.y);
    }
    if ((n & 1) && blockIdx.x == 0 && threadIdx.x == 0) out[n - 1] = (float)from_bits<half_t>(in[n - 1]);
}

// min{g : idx <= end[g]}
__device__ __forceinline__ uint32_t group_of(const uint32_t* end, uint32_t groups, uint32_t idx)
{
    uint32_t lo = 0, hi = groups - 1;
    while (lo < hi) {
        uint32_t mid = (lo + hi) >> 1;
        if (idx <= end[mid]) hi = mid; else lo = mid + 1;
    }
    return lo;
}

// Four or two elements of a row, aligned to their elements only.
typedef float Float4 __attribute__((ext_vector_type(4)));
typedef uint32_t Word2 __attribute__((ext_vector_type(2)));
typedef Float4 Float4A4 __attribute__((aligned(4)));
typedef Word2 Word2A2 __attribute__((aligned(2)));
__device__ __forceinline__ Word2 to_halves(Float4 v)
{
    half2_t a, b; a.x = (half_t)v.x; a.y = (half_t)v.y; b.x = (half_t)v.z; b.y = (half_t)v.w;
    return Word2{bits(a), bits(b)};
}
__device__ __forceinline__ Float4 to_singles(Word2 v)
{
    const half2_t a = from_bits<half2_t>(v.x), b = from_bits<half2_t>(v.y);
    return Float4{(float)a.x, (float)a.y, (float)b.x, (float)b.y};
}

// ---- scatter into grouped binary16 storage (model_init.cu:30-83) ---------------------------------
// A wavefront takes kRowsPerWave consecutive rows: their destinations are looked up by one lane each, then every load takes
// 16 bytes per lane (two rows at k = 128, four at k = 64) and all of them are in flight together.  One row at a time, each
// behind its own chain of lookups, 480k + 17.8k rows at k = 128 took 66 us per side on average to scatter and 146 to gather; this
// takes 47 and 36.
constexpr uint32_t kRowsPerWave = 16;
static inline uint32_t rows_grid(uint32_t rows, uint32_t per_wave = kRowsPerWave) { return stream_grid((uint64_t)rows * (kWave / per_wave)); }
template <int K>
__global__ __launch_bounds__(kBlock) void scatter_to_groups_kernel(const float* __restrict__ params, void* const* __restrict__ group_ptr,
                                                                  const uint32_t* __restrict__ group_end, const uint32_t* __restrict__ entity2group,
                                                                  const uint32_t* __restrict__ entity2sorted, uint32_t n, uint32_t groups)
{
    constexpr uint32_t kLanes = K / 4, kStep = kWave / kLanes, kSteps = kRowsPerWave / kStep;
    const uint32_t lane = threadIdx.x & 63u, sub = lane / kLanes, col = lane % kLanes;
    const uint64_t stride = (uint64_t)gridDim.x * kWavesPerBlock * kRowsPerWave;
    for (uint64_t base = ((uint64_t)blockIdx.x * kWavesPerBlock + (threadIdx.x >> 6)) * kRowsPerWave; base < n; base += stride) {
        Float4 v[kSteps];
#pragma unroll
        for (uint32_t j = 0; j < kSteps; ++j) {
            const uint64_t e = base + j * kStep + sub;
            if (e < n) v[j] = *reinterpret_cast<const Float4A4*>(params + e * K + col * 4);
        }
        uint64_t dst = 0;      // null: the row is in no group
        if (lane < kRowsPerWave && base + lane < n) {
            const uint32_t g = entity2group[base + lane];
            if (g < groups) {
                const uint32_t first = g ? group_end[g - 1] + 1 : 0;
                dst = reinterpret_cast<uint64_t>(group_ptr[g]) + (uint64_t)(entity2sorted[base + lane] - first) * (K * 2);
            }
        }
#pragma unroll
        for (uint32_t j = 0; j < kSteps; ++j) {
            const uint64_t to = __shfl(dst, (int)(j * kStep + sub));
            if (to) *(MF_GLOBAL Word2A2*)(to + col * 8) = to_halves(v[j]);
        }
    }
}

// ---- gather grouped storage into a dense fp32 matrix in sorted row order (mf_methods.cu:249-313) --
// Rows and lanes as in the scatter.  A lane reads 8 bytes, which is all of a binary16 row, and where there are binary32 rows
// among the wavefront's the other 8 bytes of those.  Few rows of k = 128
// are spread over more wavefronts, kRowsFew each: 5000 binary32 rows take 4.9 us instead of 5.8 with kRowsPerWave, 20001 5.5 instead of 7.3
// (one row at a time: 4.9 and 7.8).  At k = 64 both take the same (10001 rows 4.2 and 4.1), and so they do at 100k rows.
constexpr uint32_t kRowsFew = 4, kGatherFew = 24576;
template <int K, uint32_t ROWS>
__global__ __launch_bounds__(kBlock) void gather_from_groups_kernel(void* const* __restrict__ group_ptr, const uint32_t* __restrict__ group_end,
                                                                   const uint8_t* __restrict__ prec, float* __restrict__ dense, uint32_t n, uint32_t groups)
{
    constexpr uint32_t kLanes = K / 4, kStep = kWave / kLanes, kSteps = ROWS / kStep;
    const uint32_t lane = threadIdx.x & 63u, sub = lane / kLanes, col = lane % kLanes;
    const uint64_t stride = (uint64_t)gridDim.x * kWavesPerBlock * ROWS;
    for (uint64_t base = ((uint64_t)blockIdx.x * kWavesPerBlock + (threadIdx.x >> 6)) * ROWS; base < n; base += stride) {
        uint64_t src = 0;      // null: the row is in no group
        uint32_t single = 0;
        if (lane < ROWS && base + lane < n) {
            const uint32_t row = (uint32_t)(base + lane), g = group_of(group_end, groups, row);
            if (row <= group_end[g]) {
                const uint32_t local = g ? row - group_end[g - 1] - 1 : row;
                single = prec[g] ? 1u : 0u;
                src = reinterpret_cast<uint64_t>(group_ptr[g]) + (uint64_t)local * (K * 2u << single);
            }
        }
        const bool any = __ballot(single != 0u) != 0ull;
        Word2 lo[kSteps], hi[kSteps]; uint64_t from[kSteps]; uint32_t wide[kSteps];
#pragma unroll
        for (uint32_t j = 0; j < kSteps; ++j) {
            from[j] = __shfl(src, (int)(j * kStep + sub));
            wide[j] = __shfl(single, (int)(j * kStep + sub));
            if (from[j]) lo[j] = *(const MF_GLOBAL Word2A2*)(from[j] + (col * 8u << wide[j]));
        }
        if (any) {
#pragma unroll
            for (uint32_t j = 0; j < kSteps; ++j) if (wide[j]) hi[j] = *(const MF_GLOBAL Word2A2*)(from[j] + col * 16u + 8u);
        }
#pragma unroll
        for (uint32_t j = 0; j < kSteps; ++j) {
            Float4 v = to_singles(lo[j]);
            if (wide[j]) v = Float4{from_bits<float>(lo[j].x), from_bits<float>(lo[j].y), from_bits<float>(hi[j].x), from_bits<float>(hi[j].y)};
            if (from[j]) *reinterpret_cast<Float4A4*>(dense + (base + j * kStep + sub) * K + col * 4) = v;
        }
    }
}

// ---- per-group error (mf_methods.cu:327-379): one wavefront per group ---------------------------
__global__ __launch_bounds__(kWave) void group_error_kernel(float* __restrict__ grad_sum, const float* __restrict__ norm_sum, uint32_t norm_blocks,
                                                           const uint8_t* __restrict__ prec, const float* __restrict__ initial,
                                                           float* __restrict__ error_out, int k, uint32_t groups)
{
    const uint32_t g = blockIdx.x;
    if (g >= groups) return;
    const int lane = threadIdx.x;
    if (prec[g]) { if (lane == 0) error_out[g] = -1.f; return; }
    float acc = 0.f, nacc = 0.f;
    for (int e = lane; e < k; e += kWave) { const float v = grad_sum[(size_t)g * k + e]; acc += v * v; grad_sum[(size_t)g * k + e] = 0.f; }
    for (uint32_t b = lane; b < norm_blocks; b += kWave) nacc += norm_sum[(size_t)g * norm_blocks + b];
    acc = reduce_wave(acc, OpAdd());
    nacc = reduce_wave(nacc, OpAdd());
    if (lane == 0) error_out[g] = (acc / nacc) / initial[g];
}

// ---- test RMSE (rmse.h:26-189) ------------------------------------------------------------------------
// A rating's rows are read by one row of 16 lanes, 16 bytes of a binary16 row per lane at k = 128: a wavefront has four
// ratings per load and reduces four dots with four cross-lane adds.  Lane row w of a wavefront takes ratings 16 w .. 16 w + 15
// of the wavefront's 64, four at a time, so that 16 loads are in flight; a rating's values come from the lane that holds it by
// DPP broadcast within the row.
// What bounds it is the row reads, which mostly hit in L2 (test sets are sorted by user).  With one rating per wavefront
// step (one row per load, six cross-lane adds, loads waited for one rating at a time) 1.4M ratings of
// a model of 480k x 17.8k rows at k = 128, a twentieth of the groups binary32, took 261 us; this takes 70, 10 TB/s of row reads.
constexpr int kRmseBlock = 1024;
constexpr uint32_t kRmseWaves = kRmseBlock / kWave;
// One double atomic per workgroup, all on one address: two workgroups per compute unit at most.
constexpr uint32_t kRmseGrid = 512;
static inline uint32_t rmse_grid(uint32_t test_n)
{
    const uint32_t blocks = (uint32_t)(((uint64_t)test_n + kRmseBlock - 1) / kRmseBlock);
    return blocks < kRmseGrid ? blocks : kRmseGrid;
}
// Value of lane N of the same row of 16 lanes.
template <int N, class T> __device__ __forceinline__ T row_bcast(T x)
{
    return from_bits<T>((uint32_t)__builtin_amdgcn_mov_dpp((int)bits(x), 0x150 + N, 0xf, 0xf, true));
}
template <int N> __device__ __forceinline__ uint64_t row_bcast64(uint64_t x)
{
    return (uint64_t)row_bcast<N>((uint32_t)x) | ((uint64_t)row_bcast<N>((uint32_t)(x >> 32)) << 32);
}
template <int N> __device__ __forceinline__ uint64_t row_ror64(uint64_t x)
{
    return (uint64_t)row_ror<N>((uint32_t)x) | ((uint64_t)row_ror<N>((uint32_t)(x >> 32)) << 32);
}
// K / 16 elements of a row as one lane reads them: K / 8 bytes of a binary16 row, or twice as many of a binary32 row in two
// parts.  Rows are aligned to their elements only.
template <int K> struct RowPart {
    static constexpr int kWords = K / 32;
    typedef uint32_t Words __attribute__((ext_vector_type(kWords)));
    typedef Words Words2 __attribute__((aligned(2)));
    Words lo, hi;
    __device__ __forceinline__ void load_lo(uint64_t at) { lo = *(const MF_GLOBAL Words2*)at; }
    __device__ __forceinline__ void load_hi(uint64_t at) { hi = *(const MF_GLOBAL Words2*)(at + sizeof(Words)); }
    // element 2 w + b
    __device__ __forceinline__ float half_at(int w, int b) const { const half2_t h = from_bits<half2_t>(lo[w]); return b ? (float)h.y : (float)h.x; }
    __device__ __forceinline__ float single_at(int w, int b) const
    {
        const int e = 2 * w + b;
        return from_bits<float>(e < kWords ? lo[e < kWords ? e : 0] : hi[e < kWords ? 0 : e - kWords]);
    }
};
// One wavefront's rating per lane; flags: bit 0/1 the P/Q row is binary32, bit 2 there is no rating (or its id is in no group).
struct TestRating { float r; uint64_t p, q; uint32_t flags; };
// Adds the squared errors of the ratings in lanes 0 .. 3 of each lane row to acc (the same value in its 16 lanes).
template <int K, bool SINGLE> __device__ __forceinline__ void rmse_four(const TestRating& my, uint32_t lane16, double& acc)
{
    RowPart<K> a[4], b[4];
    uint64_t pa[4], qa[4]; uint32_t f[4]; float r[4];
    auto fetch = [&](auto D) {
        constexpr int d = decltype(D)::value;
        f[d] = SINGLE ? row_bcast<d>(my.flags) | 3u : row_bcast<d>(my.flags);
        r[d] = row_bcast<d>(my.r);
        pa[d] = row_bcast64<d>(my.p) + (uint64_t)(lane16 * (K / 8) << (f[d] & 1u));
        qa[d] = row_bcast64<d>(my.q) + (uint64_t)(lane16 * (K / 8) << ((f[d] >> 1) & 1u));
        a[d].load_lo(pa[d]); b[d].load_lo(qa[d]);
        if constexpr (SINGLE) { a[d].load_hi(pa[d]); b[d].load_hi(qa[d]); }
    };
    fetch(std::integral_constant<int, 0>()); fetch(std::integral_constant<int, 1>());
    fetch(std::integral_constant<int, 2>()); fetch(std::integral_constant<int, 3>());
    const bool any = SINGLE || __ballot(((f[0] | f[1] | f[2] | f[3]) & 3u) != 0u) != 0ull;
    if (!SINGLE && any) {
#pragma unroll
        for (int d = 0; d < 4; ++d) {
            if (f[d] & 1u) a[d].load_hi(pa[d]); else a[d].hi = a[d].lo;
            if (f[d] & 2u) b[d].load_hi(qa[d]); else b[d].hi = b[d].lo;
        }
    }
#pragma unroll
    for (int d = 0; d < 4; ++d) {
        float dot = 0.f;
        if (any) {
#pragma unroll
            for (int w = 0; w < RowPart<K>::kWords; ++w)
#pragma unroll
                for (int e = 0; e < 2; ++e)
                    dot = __builtin_fmaf(SINGLE || (f[d] & 1u) ? a[d].single_at(w, e) : a[d].half_at(w, e),
                                         SINGLE || (f[d] & 2u) ? b[d].single_at(w, e) : b[d].half_at(w, e), dot);
        } else {
#pragma unroll
            for (int w = 0; w < RowPart<K>::kWords; ++w)
#pragma unroll
                for (int e = 0; e < 2; ++e) dot = __builtin_fmaf(a[d].half_at(w, e), b[d].half_at(w, e), dot);
        }
        dot = reduce_row16(dot, OpAdd());
        const double err = f[d] & 4u ? 0.0 : (double)(r[d] - dot);
        acc += err * err;
    }
}
// All ratings of a wavefront.  A lane without a rating reads the rows of one that has, and adds nothing.
template <int K, bool SINGLE> __device__ __forceinline__ void rmse_wave(TestRating my, double& acc)
{
    const uint64_t valid = __ballot(!(my.flags & 4u));
    if (!valid) return;
    const int some = __builtin_ctzll(valid);
    const uint64_t p = bcast(my.p, some), q = bcast(my.q, some); const uint32_t f = bcast(my.flags, some);
    if (my.flags & 4u) { my.p = p; my.q = q; my.flags = f | 4u; }
    const uint32_t lane16 = threadIdx.x & 15u;
    // up to four ratings lie in the first batch: one takes 4.7 us (grouped, k = 128) instead of 5.7
    const int batches = valid & ~0x000f000f000f000full ? 4 : 1;
    // not unrolled: four batches' loads in flight at once would not fit the registers of 16 wavefronts per compute unit
#pragma unroll 1
    for (int batch = 0; batch < batches; ++batch) {
        rmse_four<K, SINGLE>(my, lane16, acc);
        my.r = row_ror<4>(my.r); my.flags = row_ror<4>(my.flags);
        my.p = row_ror64<4>(my.p); my.q = row_ror64<4>(my.q);
    }
}
__device__ __forceinline__ void rmse_block_sum(double acc, double* out)
{
    __shared__ double part[kRmseWaves * 4];
    if ((threadIdx.x & 15u) == 0u) part[threadIdx.x >> 4] = acc;
    __syncthreads();
    if (threadIdx.x == 0) {
        double s = 0;
        for (uint32_t i = 0; i < kRmseWaves * 4; ++i) s += part[i];
        atomicAdd(out, s);
    }
}

template <int K>
__global__ __launch_bounds__(kRmseBlock) void rmse_dense_kernel(const mf_node* __restrict__ test, uint32_t test_n, const float* __restrict__ P,
                                                               const float* __restrict__ Q, double* sum_sq)
{
    const uint32_t lane = threadIdx.x & 63u;
    double acc = 0;
    for (uint64_t base = ((uint64_t)(threadIdx.x >> 6) * gridDim.x + blockIdx.x) * kWave; base < test_n; base += (uint64_t)gridDim.x * kRmseBlock) {
        TestRating my = {0.f, 0, 0, 7u};
        if (base + lane < test_n) {
            const Rating x = load_rating(test, (uint32_t)(base + lane));
            my = {x.r, reinterpret_cast<uint64_t>(P) + (uint64_t)x.u * (K * 4u), reinterpret_cast<uint64_t>(Q) + (uint64_t)x.v * (K * 4u), 3u};
        }
        rmse_wave<K, true>(my, acc);
    }
    rmse_block_sum(acc, sum_sq);
}

template <int K>
__global__ __launch_bounds__(kRmseBlock) void rmse_grouped_kernel(const mf_node* __restrict__ test, uint32_t test_n, void* const* __restrict__ p, void* const* __restrict__ q,
                                                                 const uint32_t* __restrict__ user_end, const uint32_t* __restrict__ item_end,
                                                                 const uint8_t* __restrict__ user_prec, const uint8_t* __restrict__ item_prec,
                                                                 uint32_t user_groups, uint32_t item_groups, double* sum_sq)
{
    extern __shared__ __align__(16) uint8_t smem[];
    uint64_t* pptr_s = reinterpret_cast<uint64_t*>(smem);
    uint64_t* qptr_s = pptr_s + user_groups;
    uint32_t* uend_s = reinterpret_cast<uint32_t*>(qptr_s + item_groups);
    uint32_t* iend_s = uend_s + user_groups;
    uint8_t* uprec_s = reinterpret_cast<uint8_t*>(iend_s + item_groups);
    uint8_t* iprec_s = uprec_s + user_groups;
    for (uint32_t g = threadIdx.x; g < user_groups; g += blockDim.x) { pptr_s[g] = reinterpret_cast<uint64_t>(p[g]); uend_s[g] = user_end[g]; uprec_s[g] = user_prec[g]; }
    for (uint32_t g = threadIdx.x; g < item_groups; g += blockDim.x) { qptr_s[g] = reinterpret_cast<uint64_t>(q[g]); iend_s[g] = item_end[g]; iprec_s[g] = item_prec[g]; }
    __syncthreads();
    const uint32_t lane = threadIdx.x & 63u;
    double acc = 0;
    for (uint64_t base = ((uint64_t)(threadIdx.x >> 6) * gridDim.x + blockIdx.x) * kWave; base < test_n; base += (uint64_t)gridDim.x * kRmseBlock) {
        TestRating my = {0.f, 0, 0, 4u};
        if (base + lane < test_n) {
            const Rating x = load_rating(test, (uint32_t)(base + lane));
            const uint32_t ug = group_of(uend_s, user_groups, x.u), ig = group_of(iend_s, item_groups, x.v);
            if (x.u <= uend_s[ug] && x.v <= iend_s[ig]) {
                const uint32_t urow = ug ? x.u - uend_s[ug - 1] - 1 : x.u;
                const uint32_t irow = ig ? x.v - iend_s[ig - 1] - 1 : x.v;
                const uint32_t up = uprec_s[ug] ? 1u : 0u, ip = iprec_s[ig] ? 1u : 0u;
                my = {x.r, pptr_s[ug] + (uint64_t)urow * (K * (up ? 4u : 2u)), qptr_s[ig] + (uint64_t)irow * (K * (ip ? 4u : 2u)), up | (ip << 1)};
            }
        }
        rmse_wave<K, false>(my, acc);
    }
    rmse_block_sum(acc, sum_sq);
}

// ---- model init (model_init.cu:19-28): N(0,1)*0.01 from counter-derived bits ----------------------
// ln x, x in (0,1], from +,-,*,/ only (identical bits on any IEEE machine).
__device__ __forceinline__ double det_log(double x)
{
    const uint64_t b = __builtin_bit_cast(uint64_t, x);
    int e = (int)((b >> 52) & 0x7ff) - 1022;
    double m = __builtin_bit_cast(double, (b & 0x000fffffffffffffull) | 0x3fe0000000000000ull);
    if (m < 0.70710678118654752440) { m = m * 2.0; e = e - 1; }
    const double s = (m - 1.0) / (m + 1.0);
    const double s2 = s * s;
    double acc = 1.0 / 21.0;
    acc = acc * s2 + 1.0 / 19.0;
    acc = acc * s2 + 1.0 / 17.0;
    acc = acc * s2 + 1.0 / 15.0;
    acc = acc * s2 + 1.0 / 13.0;
    acc = acc * s2 + 1.0 / 11.0;
    acc = acc * s2 + 1.0 / 9.0;
    acc = acc * s2 + 1.0 / 7.0;
    acc = acc * s2 + 1.0 / 5.0;
    acc = acc * s2 + 1.0 / 3.0;
    acc = acc * s2 + 1.0;
    const double lnm = (2.0 * s) * acc;
    return (double)e * 0.69314718055994530942 + lnm;
}
__device__ __forceinline__ double det_cos2pi(double t)
{
    const double t4 = t * 4.0;
    const int q = (int)t4;
    const double f = t4 - (double)q;
    const double a = f * 1.57079632679489661923;
    const double a2 = a * a;
    double c = 1.0 / 2432902008176640000.0;
    c = -1.0 / 6402373705728000.0 + a2 * c;
    c = 1.0 / 20922789888000.0 + a2 * c;
    c = -1.0 / 87178291200.0 + a2 * c;
    c = 1.0 / 479001600.0 + a2 * c;
    c = -1.0 / 3628800.0 + a2 * c;
    c = 1.0 / 40320.0 + a2 * c;
    c = -1.0 / 720.0 + a2 * c;
    c = 1.0 / 24.0 + a2 * c;
    c = -1.0 / 2.0 + a2 * c;
    c = 1.0 + a2 * c;
    double s = 1.0 / 51090942171709440000.0;
    s = -1.0 / 121645100408832000.0 + a2 * s;
    s = 1.0 / 355687428096000.0 + a2 * s;
    s = -1.0 / 1307674368000.0 + a2 * s;
    s = 1.0 / 6227020800.0 + a2 * s;
    s = -1.0 / 39916800.0 + a2 * s;
    s = 1.0 / 362880.0 + a2 * s;
    s = -1.0 / 5040.0 + a2 * s;
    s = 1.0 / 120.0 + a2 * s;
    s = -1.0 / 6.0 + a2 * s;
    s = 1.0 + a2 * s;
    s = a * s;
    switch (q & 3) { case 0: return c; case 1: return -s; case 2: return -c; default: return s; }
}
// N(0,1) from 64 bits (Box-Muller over the two 32-bit halves)
__device__ __forceinline__ double det_normal(uint64_t h)
{
    const uint32_t a = (uint32_t)(h >> 32), b = (uint32_t)h;
    const double u1 = ((double)a + 1.0) * 2.3283064365386962890625e-10;
    const double u2 = (double)b * 2.3283064365386962890625e-10;
    const double rad = __builtin_sqrt(-2.0 * det_log(u1));
    return rad * det_cos2pi(u2);
}
__global__ __launch_bounds__(kStreamBlock) void init_normal_kernel(float* __restrict__ out, uint64_t n, uint64_t base, double scale)
{
    const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride)
        out[i] = (float)(det_normal(mix64(base ^ i)) * scale);
}

// ---- seeded synthetic ratings (mf_generate_ratings) ------------------------------------------------
struct SynthTables {
    const double* user_cdf; const double* item_cdf;       // cumulative Zipf weights, last entry 1.0
    const uint32_t* user_perm; const uint32_t* item_perm; // popularity rank -> id
    const float* U; const float* V;                       // [rows][rank] factors, or null (bimodal)
};
// smallest index whose cumulative weight exceeds x (x in [0,1), cdf[count-1] = 1)
__device__ __forceinline__ uint32_t cdf_rank(const double* cdf, uint32_t count, double x)
{
    uint32_t lo = 0, hi = count - 1;
    while (lo < hi) {
        const uint32_t mid = (lo + hi) >> 1;
        if (x < cdf[mid]) hi = mid; else lo = mid + 1;
    }
    return lo;
}
__global__ __launch_bounds__(kStreamBlock) void generate_ratings_kernel(mf_synth_config c, SynthTables t, uint64_t key, uint64_t first, uint64_t count,
                                                                      float inv_step, mf_node* __restrict__ out)
{
    const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < count; i += stride) {
        const uint64_t j = first + i;
        const double xu = (double)(mix64(key ^ (j * 4 + 0)) >> 11) * 1.1102230246251565404e-16;      // 53 bits in [0,1)
        const double xi = (double)(mix64(key ^ (j * 4 + 1)) >> 11) * 1.1102230246251565404e-16;
        const uint32_t u = t.user_perm[cdf_rank(t.user_cdf, c.n_users, xu)];
        const uint32_t v = t.item_perm[cdf_rank(t.item_cdf, c.n_items, xi)];
        const float nz = (float)(det_normal(mix64(key ^ (j * 4 + 2))) * (double)c.noise);
        float r;
        if (c.bimodal) {
            const double xm = (double)(mix64(key ^ (j * 4 + 3)) >> 11) * 1.1102230246251565404e-16;
            const float m = xm < 0.5 ? 20.0f : 80.0f;
            r = fminf(fmaxf(roundf(m + nz), c.lo), c.hi) * 0.04f + 1.0f;
        } else {
            float dot = 0.0f;
            for (uint32_t k = 0; k < c.rank; ++k) dot = dot + t.U[(size_t)u * c.rank + k] * t.V[(size_t)v * c.rank + k];
            const float val = (dot + c.mean) + nz;
            r = fminf(fmaxf(roundf(val * inv_step) * c.step, c.lo), c.hi);
        }
        out[i].r = r; out[i].u = u; out[i].i = v;
    }
}

// ---- preprocessing (preprocess_utils.h:6-36) ---------------------------------------------------
__global__ __launch_bounds__(kStreamBlock) void iota_kernel(uint32_t* __restrict__ a, uint32_t n)
{
    const uint32_t stride = gridDim.x * blockDim.x;
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) a[i] = i;
}
// user_item_histogram (preprocess_utils.h:13-19).  Global atomics on scattered counters go to the memory side one by one, and with
// Zipf-like popularity a few counters would take percents of them, so ids are counted in LDS first.  Three ways:
//   few     up to kHistFew ratings: a workgroup counts its ratings in a hash table, kHistFewLog bits of (id, count) slots per side, a
//           slot claimed by the first id that hashes to it (two probes); ids that find both taken go to memory, and the table
//           follows at the end.
//   ranges  a workgroup counts one range of ids, over one chunk of the ratings.  User and item ids are laid end to end and cut
//           into ranges of kHistBins; the workgroups of one chunk sit on one XCD, so that its L2 hands them the same ratings.  How
//           far the ids reach is not an argument: every workgroup takes the largest ids of the same kHistSample ratings, spread over
//           the input, and the few above them are added in memory by the workgroups of the first and the last range.
//   hashed  as few, with tables twice as large on one workgroup per compute unit: ids that reach past kHistRanges ranges, or past
//           kHistSure while few different ones make up most of the ratings (or there are less than kHistSampled ratings).
// What bounds the ranges is a workgroup's pass over its chunk (L1 and the instructions per id), so their time follows
// ratings / chunks: 100M ratings take 0.46 ms in 3 ranges, 0.81 in 7 (1.63 without the next tile's loads in flight), 1.55 in 15,
// 2.95 from 17 to 32, up to a fifth more under Zipf(1.2).  A workgroup with ids of both sides makes two passes and the others wait
// for it: 50M ratings of 1M + 200k ids took 1.67 ms in 15 ranges with one such and take 0.81 in 16 without.  (Calls repeated on the same
// ratings; the one call of a training run on 100M ratings, 7 ranges, takes 1.1 ms under the profiler.)  In front of that come 13 to
// 20 us: 160 KB of counters cleared, the sample, the counters' way to memory.
// The tables' time follows the ids that find no slot.  50M ratings of 1M + 625k ids (21 ranges), hashed / ranges: flat 3.69 / 1.54 ms,
// Zipf(0.8) 3.10 / 1.54, Zipf(1.0) 1.79 / 1.53, Zipf(1.1) 1.12 / 1.54, Zipf(1.2) 0.68 / 1.54.  The sample tells them apart: 7942, 6980,
// 4653, 3441 and 2341 different hash values of both sides, and the line is at kHistDistinct.  With few ratings the tables are the
// faster way for flat ids, too: 39 / 49 us at 400k, 54 / 49 at 600k.
// Up to kHistFew ratings the same goes for fewer ids: 100k ratings of 480k + 17.8k ids take 14 us (flat) and 8 (Zipf(1.2)), where the
// ranges took 27, one rating 4 instead of 14 to 21.  At 200k ratings the tables' lead is 18 to 21 against 22 us there, but with up
// to 5k ids, where all tables add to the same few counters, they take 38 to 56 against 13 to 16.  For the sake of these the
// workgroups are few, too: with 128 instead of kHistFewGrid 100k ratings of 1000 + 500 ids took 29 us instead of 13, at 1 to 3 us
// less where there are many ids.
//
// Counters of a range are 16 bits wide, twice as many ids per range.  The thread that brings one to 2^15 moves 2^15 to memory; it has done
// so before the next barrier, and between two barriers there are kHistBlock * kHistUnroll = 2^14 ids per side at most.
constexpr int kHistBlock = 1024;
constexpr uint32_t kHistUnroll = 16;
constexpr uint32_t kHistHalf = 40448, kHistBins = 2 * kHistHalf;      // words, each the counters of ids x and x + kHistHalf of the range
constexpr uint32_t kHistGrid = 256, kHistPerXcd = kHistGrid / kXcds;  // one workgroup per compute unit
constexpr uint32_t kHistRanges = kHistPerXcd, kHistSure = 16, kHistDistinct = 4000;
constexpr uint32_t kHistSampled = 1u << 19;
constexpr uint32_t kHistLog = 13, kHistSlots = 1u << kHistLog, kHistHashedMin = 4096;      // ratings of a workgroup
constexpr uint32_t kHistFew = 1u << 17, kHistFewLog = 12, kHistFewGrid = 32;
constexpr uint32_t kHistSample = 4 * kHistBlock, kHistSeenBits = 16;
constexpr uint32_t kHistChunkMin = 1u << 14;                          // ratings
constexpr size_t kHistLds = (size_t)kHistHalf * 4;
static_assert(4 * kHistSlots <= kHistHalf && (2u << kHistSeenBits) / 32 <= kHistHalf, "the hash tables and the sample's bits fit where the counters are");
static_assert(kHistBlock * kHistUnroll + 0x8000u < 0x10000u, "a 16-bit counter cannot overflow between two barriers");
struct HistogramRange {
    uint32_t* bin;            // LDS
    uint32_t lo, size;        // ids [lo, lo + size) of this side are this workgroup's
    uint32_t at;              // first counter
    uint32_t known;           // ids from here on are in no range
    uint32_t* global_bin;
    bool rest;                // this workgroup takes those
    // kHistUnroll ids of this lane, of which the first `mine` count.  All adds are issued before the first result is looked at,
    // and then all results at once: adding 0x400 to both halves of a word sets a top bit from 0x7c00 on.
    __device__ __forceinline__ void count(const uint32_t (&id)[kHistUnroll], uint32_t mine) const
    {
        uint32_t old[kHistUnroll], x[kHistUnroll], high = 0, largest = 0;
#pragma unroll
        for (uint32_t j = 0; j < kHistUnroll; ++j) x[j] = id[j] - lo;
        if (__ballot(mine != kHistUnroll)) {
#pragma unroll
            for (uint32_t j = 0; j < kHistUnroll; ++j) if (j >= mine) x[j] = 0xffffffffu;
        }
#pragma unroll
        for (uint32_t j = 0; j < kHistUnroll; ++j) {
            const uint32_t c = at + x[j];
            old[j] = 0u;
            if (x[j] < size) old[j] = atomicAdd(&bin[c < kHistHalf ? c : c - kHistHalf], c < kHistHalf ? 1u : 0x10000u);
        }
#pragma unroll
        for (uint32_t j = 0; j < kHistUnroll; ++j) { high |= old[j] + 0x04000400u; largest = max(largest, id[j]); }
        if (!(high & 0x80008000u) && !(rest && largest >= known)) return;
#pragma unroll
        for (uint32_t j = 0; j < kHistUnroll; ++j) {
            const uint32_t c = at + x[j];
            if (x[j] < size) {
                if (((c < kHistHalf ? old[j] << 16 : old[j]) >> 16) != 0x7fffu) continue;
                atomicSub(&bin[c < kHistHalf ? c : c - kHistHalf], c < kHistHalf ? 0x8000u : 0x80000000u);
                atomicAdd(&global_bin[id[j]], 0x8000u);
            } else if (rest && j < mine && id[j] >= known) atomicAdd(&global_bin[id[j]], 1u);
        }
    }
};
template <uint32_t LOG> __device__ __forceinline__ void hashed_count(uint32_t* tag, uint32_t* cnt, uint32_t id, uint32_t* global_bin)
{
    uint32_t s = (id * 2654435761u) >> (32 - LOG);
#pragma unroll
    for (int probe = 0; probe < 2; ++probe, s ^= 1u) {
        uint32_t t = tag[s];
        if (t == 0u) t = atomicCAS(&tag[s], 0u, id + 1u);
        if (t == 0u || t == id + 1u) { atomicAdd(&cnt[s], 1u); return; }
    }
    atomicAdd(&global_bin[id], 1u);
}
// Ratings [begin, end), AHEAD of each lane in flight.  tab: 4 << LOG words of LDS, zero: user tags, user counts, item tags, item counts.
template <uint32_t LOG, uint32_t AHEAD>
__device__ __forceinline__ void histogram_hashed(const mf_node* __restrict__ R, uint64_t begin, uint64_t end, uint32_t* user_bin, uint32_t* item_bin, uint32_t* tab)
{
    uint32_t* utag = tab, *ucnt = tab + (1u << LOG), *itag = tab + (2u << LOG), *icnt = tab + (3u << LOG);
    for (uint64_t base = begin; base < end; base += kHistBlock * AHEAD) {
        const uint32_t* w = reinterpret_cast<const uint32_t*>(R + base);
        const uint32_t left = end - base < kHistBlock * AHEAD ? (uint32_t)(end - base) : kHistBlock * AHEAD;
        uint32_t u[AHEAD], v[AHEAD];
#pragma unroll
        for (uint32_t j = 0; j < AHEAD; ++j) {
            const uint32_t o = min(j * kHistBlock + threadIdx.x, left - 1u) * 3u;
            u[j] = __builtin_nontemporal_load(w + o + 1u); v[j] = __builtin_nontemporal_load(w + o + 2u);
        }
#pragma unroll
        for (uint32_t j = 0; j < AHEAD; ++j) {
            if (j * kHistBlock + threadIdx.x >= left) continue;
            hashed_count<LOG>(utag, ucnt, u[j], user_bin);
            hashed_count<LOG>(itag, icnt, v[j], item_bin);
        }
    }
    __syncthreads();
    for (uint32_t s = threadIdx.x; s < (1u << LOG); s += kHistBlock) {
        if (utag[s]) atomicAdd(&user_bin[utag[s] - 1u], ucnt[s]);
        if (itag[s]) atomicAdd(&item_bin[itag[s] - 1u], icnt[s]);
    }
}
__global__ __launch_bounds__(kHistBlock) void histogram_few_kernel(const mf_node* __restrict__ R, uint32_t n, uint32_t per_block, uint32_t* user_bin, uint32_t* item_bin)
{
    __shared__ uint32_t tab[4u << kHistFewLog];
    for (uint32_t i = threadIdx.x; i < 4u << kHistFewLog; i += kHistBlock) tab[i] = 0u;
    __syncthreads();
    const uint64_t begin = (uint64_t)blockIdx.x * per_block, end = begin + per_block;
    histogram_hashed<kHistFewLog, 4>(R, begin, end < n ? end : n, user_bin, item_bin, tab);
}
__global__ __launch_bounds__(kHistBlock) void histogram_kernel(const mf_node* __restrict__ R, uint32_t n, uint32_t* user_bin, uint32_t* item_bin)
{
    extern __shared__ uint32_t hist_bin[];
    __shared__ uint32_t reach[2], distinct;
    uint32_t su[kHistSample / kHistBlock], sv[kHistSample / kHistBlock];
#pragma unroll
    for (uint32_t j = 0; j < kHistSample / kHistBlock; ++j) {
        const uint32_t at = (uint32_t)((uint64_t)n * (j * kHistBlock + threadIdx.x) / kHistSample);
        su[j] = R[at].u; sv[j] = R[at].i;
    }
    if (threadIdx.x < 2) reach[threadIdx.x] = 0u;
    if (threadIdx.x == 0) distinct = 0u;
    for (uint32_t i = threadIdx.x; i < kHistHalf; i += kHistBlock) hist_bin[i] = 0u;      // while the sample is on its way
    __syncthreads();
    uint32_t mu = 0, mv = 0;
#pragma unroll
    for (uint32_t j = 0; j < kHistSample / kHistBlock; ++j) { mu = max(mu, su[j]); mv = max(mv, sv[j]); }
    for (int d = kWave / 2; d; d >>= 1) { mu = max(mu, (uint32_t)__shfl_xor((int)mu, d)); mv = max(mv, (uint32_t)__shfl_xor((int)mv, d)); }
    if ((threadIdx.x & 63u) == 0u) { atomicMax(&reach[0], mu); atomicMax(&reach[1], mv); }
    __syncthreads();
    const uint32_t most = (kHistRanges + 1u) * kHistBins;
    const uint32_t users = (uint32_t)__builtin_amdgcn_readfirstlane((int)min(reach[0], most - 1u)) + 1u;
    const uint32_t items = (uint32_t)__builtin_amdgcn_readfirstlane((int)min(reach[1], most - 1u)) + 1u;
    const uint32_t user_ranges = (users + kHistBins - 1u) / kHistBins, apart = user_ranges + (items + kHistBins - 1u) / kHistBins;
    const uint32_t together = (users + items + kHistBins - 1u) / kHistBins;
    bool hashed = together > kHistRanges || (together > kHistSure && n < kHistSampled);
    if (!hashed && together > kHistSure) {
        // how many different ids the sample has: a bit per side and hash value, counted and cleared
        constexpr uint32_t kWords = (1u << kHistSeenBits) / 32;
#pragma unroll
        for (uint32_t j = 0; j < kHistSample / kHistBlock; ++j) {
            const uint32_t hu = (su[j] * 2654435761u) >> (32 - kHistSeenBits), hv = (sv[j] * 2654435761u) >> (32 - kHistSeenBits);
            atomicOr(&hist_bin[hu / 32u], 1u << (hu % 32u));
            atomicOr(&hist_bin[kWords + hv / 32u], 1u << (hv % 32u));
        }
        __syncthreads();
        uint32_t count = 0;
        for (uint32_t i = threadIdx.x; i < 2u * kWords; i += kHistBlock) { count += (uint32_t)__popc(hist_bin[i]); hist_bin[i] = 0u; }
        for (int d = kWave / 2; d; d >>= 1) count += (uint32_t)__shfl_xor((int)count, d);
        if ((threadIdx.x & 63u) == 0u) atomicAdd(&distinct, count);
        __syncthreads();
        hashed = distinct < kHistDistinct;
    }
    if (hashed) {
        const uint32_t blocks = min(kHistGrid, n / kHistHashedMin + 1u);
        if (blockIdx.x < blocks) histogram_hashed<kHistLog, 8>(R, (uint64_t)n * blockIdx.x / blocks, (uint64_t)n * (blockIdx.x + 1u) / blocks, user_bin, item_bin, hist_bin);
        return;
    }
    // The items begin a range of their own unless the one more range takes half of the chunks
    const bool split = apart == together || (apart <= kHistPerXcd && 2u * (kHistPerXcd / apart) > kHistPerXcd / together);
    const uint32_t ranges = split ? apart : together, item_base = split ? user_ranges * kHistBins : users;
    const uint32_t xcd = blockIdx.x % kXcds, local = blockIdx.x / kXcds;
    const uint32_t per_xcd = kHistPerXcd / ranges, by_size = n / kHistChunkMin + 1u;
    const uint32_t chunks = min(per_xcd * kXcds, by_size), chunk = xcd + kXcds * (local / ranges);
    if (local / ranges >= per_xcd || chunk >= chunks) return;
    const uint32_t first = local % ranges * kHistBins, last = first + kHistBins;
    const HistogramRange U = {hist_bin, first, first < users ? min(last, users) - first : 0u, 0u, users, user_bin, first == 0u};
    const uint32_t ilo = first > item_base ? first - item_base : 0u;
    const HistogramRange I = {hist_bin, ilo, last > item_base ? min(last - item_base, items) - ilo : 0u, U.size, items, item_bin, last >= item_base + items};
    const uint32_t begin = (uint32_t)((uint64_t)n * chunk / chunks), end = (uint32_t)((uint64_t)n * (chunk + 1u) / chunks);
    constexpr uint32_t kTile = kHistBlock * kHistUnroll;
    // field: 1 the users, 2 the items
    auto sweep = [&](const HistogramRange& range, uint32_t field) {
        uint32_t next[kHistUnroll];
        auto fetch = [&](uint64_t tile) {
            if (tile >= end) return;
            const uint32_t* w = reinterpret_cast<const uint32_t*>(R + tile) + field;
            const uint32_t most = end - tile < kTile ? (uint32_t)(end - tile) - 1u : kTile - 1u;
#pragma unroll
            for (uint32_t j = 0; j < kHistUnroll; ++j) next[j] = w[min(j * kHistBlock + threadIdx.x, most) * 3u];
        };
        fetch(begin);
        for (uint64_t tile = begin; tile < end; tile += kTile) {
            uint32_t id[kHistUnroll];
#pragma unroll
            for (uint32_t j = 0; j < kHistUnroll; ++j) id[j] = next[j];
            fetch(tile + kTile);        // on their way while these are counted
            const uint32_t left = end - tile < kTile ? (uint32_t)(end - tile) : kTile;
            const uint32_t mine = left <= threadIdx.x ? 0u : (left - threadIdx.x + kHistBlock - 1u) / kHistBlock;
            range.count(id, mine);
            __syncthreads();
        }
    };
    if (U.size) sweep(U, 1u);
    if (I.size) sweep(I, 2u);
    for (uint32_t c = threadIdx.x; c < U.size + I.size; c += kHistBlock) {
        const uint32_t count = c < kHistHalf ? hist_bin[c] & 0xffffu : hist_bin[c - kHistHalf] >> 16;
        if (count) atomicAdd(c < U.size ? &user_bin[U.lo + c] : &item_bin[I.lo + (c - U.size)], count);
    }
}
// The ratings as a stream of words, four per lane and load: word w is a rating value, a user or an item by w % 3 (for the
// words of the t-th four: (t + j) % 3), and the values go back with the ids around them, so that whole lines are read and written.
// What bounds it is the lookups, a line each.  With a thread per rating, two strided loads and two strided stores, 100M ratings
// took 1.25 ms; this takes 1.05, 200M lookups that fetch 12 TB/s of lines from the L2.
// UNROLL: fours of a lane whose lookups are in flight together.  While the lanes are few, more of them are better than more lookups
// per lane: one against four, 100k ratings of 5M + 1M ids take 5 us instead of 7, 800k of 480k + 17.8k ids 7.9 instead of 8.7, 1.3M 12.4
// instead of 11.9.
typedef uint32_t Word4 __attribute__((ext_vector_type(4)));
typedef Word4 Word4A4 __attribute__((aligned(4)));
template <uint32_t UNROLL>
__global__ __launch_bounds__(kStreamBlock, 8) void reindex_kernel(uint32_t* R, const uint32_t* __restrict__ user2sorted, const uint32_t* __restrict__ item2sorted, uint64_t words)
{
    const uint64_t fours = words / 4, stride = (uint64_t)gridDim.x * kStreamBlock * UNROLL;
    Word4A4* to = reinterpret_cast<Word4A4*>(R);
    for (uint64_t base = (uint64_t)blockIdx.x * kStreamBlock * UNROLL + threadIdx.x; base < fours; base += stride) {
        Word4 x[UNROLL], y[UNROLL];
#pragma unroll
        for (uint32_t i = 0; i < UNROLL; ++i) {
            x[i] = Word4{0u, 0u, 0u, 0u};
            if (base + i * kStreamBlock < fours) x[i] = __builtin_nontemporal_load(to + base + i * kStreamBlock);
        }
        // no branches, which would wait for one lookup before the next: a lane with nothing to look up reads entry 0
#pragma unroll
        for (uint32_t i = 0; i < UNROLL; ++i) {
            const uint64_t t = base + i * kStreamBlock;
            const uint32_t kind = (uint32_t)(t % 3u);
#pragma unroll
            for (uint32_t j = 0; j < 4; ++j) {
                const uint32_t word = kind + j % 3u, id = word % 3u && t < fours ? x[i][j] : 0u;      // word < 5
                y[i][j] = (word == 2u ? item2sorted : user2sorted)[id];
                if (word % 3u == 0u) y[i][j] = x[i][j];
            }
        }
#pragma unroll
        for (uint32_t i = 0; i < UNROLL; ++i)
            if (base + i * kStreamBlock < fours) __builtin_nontemporal_store(y[i], to + base + i * kStreamBlock);
    }
    const uint64_t w = fours * 4 + threadIdx.x;      // up to three words are left
    if (blockIdx.x == 0 && w < words && w % 3u) R[w] = (w % 3u == 1u ? user2sorted : item2sorted)[R[w]];
}

static size_t group_table_lds(uint32_t ug, uint32_t ig) { return (size_t)(ug + ig) * (8 + 4 + 1) + 16; }

}  // namespace mf

using namespace mf;

// ---- access-pattern probe ------------------------------------------------------------------------
// The memory traffic of one epoch of updates without the arithmetic: per rating the two rows are read and, where
// the hot-row tables keep the update, written back unchanged (the loaded value plus `zero`, a kernel argument the
// compiler cannot fold).  The same draw as the update kernels' thinning decides; a kept update of a hot row is a
// store here too.  What it sustains is the ceiling the memory system sets for this sequence of addresses and this
// write policy, the figure the update kernels' epoch time is compared with.
template <int BYTES, bool COH, int BYTES_Q = BYTES>       // bytes per lane and side: a row is 64 * BYTES bytes
__global__ __launch_bounds__(kBlock) void row_traffic_probe_kernel(const mf_node* R, uint32_t n, uint8_t* P, uint8_t* Q, uint32_t per_worker,
                                                                  const uint8_t* keep_u, const uint8_t* keep_v, const uint16_t* slot_u, const uint16_t* slot_v,
                                                                  uint32_t slots_u, uint32_t slots_v, uint8_t* RP, uint8_t* RQ, uint64_t key, uint32_t zero)
{
    using T = typename std::conditional<BYTES == 8, uint64_t, typename std::conditional<BYTES == 4, uint32_t, uint16_t>::type>::type;
    using TQ = typename std::conditional<BYTES_Q == 8, uint64_t, typename std::conditional<BYTES_Q == 4, uint32_t, uint16_t>::type>::type;
    constexpr int kDepth = 4;
    const int lane = threadIdx.x & (kWave - 1);
    const uint32_t worker = blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
    const uint64_t begin64 = (uint64_t)worker * per_worker;
    if (begin64 >= n) return;
    const uint32_t xcd = xcd_id();
    const uint32_t begin = (uint32_t)begin64, end = (uint64_t)begin + per_worker < n ? begin + per_worker : n;
    for (uint32_t base = begin; base < end; base += kWave) {
        uint32_t mu = 0, mv = 0, keep = 0;      // keep: bit0/bit1 write the P/Q row back, bit2/bit3 the row is this XCD's copy of a replicated row
        if (base + (uint32_t)lane < end) {
            const Rating x = load_rating(R, base + (uint32_t)lane);
            mu = x.u; mv = x.v; keep = 3u;
            if (keep_u) {
                const uint32_t rnd = (uint32_t)(mix64(key ^ (((uint64_t)(base + (uint32_t)lane) << 20) ^ (uint64_t)worker ^ 0x7468696eull)) >> 40);
                const uint32_t ku = keep_u[mu], kv = keep_v[mv];
                if (ku == kKeepReplicated || ku == kKeepReplicatedAdded) { keep |= 4u; mu = xcd * slots_u + slot_u[mu]; }
                else if (ku != 255u && (((rnd & 0xfffu) * 255u) >> 12) > ku) keep &= ~1u;
                if (kv == kKeepReplicated || kv == kKeepReplicatedAdded) { keep |= 8u; mv = xcd * slots_v + slot_v[mv]; }
                else if (kv != 255u && (((rnd >> 12) * 255u) >> 12) > kv) keep &= ~2u;
            }
        }
        const int cnt = end - base < (uint32_t)kWave ? (int)(end - base) : kWave;
        for (int j0 = 0; j0 < cnt; j0 += kDepth) {
            T a[kDepth]; TQ b[kDepth]; T* pa[kDepth]; TQ* pb[kDepth]; uint32_t kp[kDepth];
#pragma unroll
            for (int d = 0; d < kDepth; ++d) {
                const int j = j0 + d < cnt ? j0 + d : cnt - 1;
                kp[d] = j0 + d < cnt ? bcast(keep, j) : 0u;
                const uint32_t flags = bcast(keep, j);
                pa[d] = reinterpret_cast<T*>(((flags & 4u) ? RP : P) + (size_t)bcast(mu, j) * (kWave * BYTES)) + lane;
                pb[d] = reinterpret_cast<TQ*>(((flags & 8u) ? RQ : Q) + (size_t)bcast(mv, j) * (kWave * BYTES_Q)) + lane;
                a[d] = row_load(pa[d]); b[d] = row_load(pb[d]);
            }
#pragma unroll
            for (int d = 0; d < kDepth; ++d) {
                if (kp[d] & 4u) row_store<false>(pa[d], (T)(a[d] + (T)zero)); else if (kp[d] & 1u) row_store<COH>(pa[d], (T)(a[d] + (T)zero));
                if (kp[d] & 8u) row_store<false>(pb[d], (TQ)(b[d] + (TQ)zero)); else if (kp[d] & 2u) row_store<COH>(pb[d], (TQ)(b[d] + (TQ)zero));
            }
        }
    }
}

namespace {
// cumulative weights (rank+1)^-alpha, normalised by their sum; summed in rank order in double
std::vector<double> zipf_cdf(uint32_t count, float alpha)
{
    std::vector<double> cdf(count);
    double sum = 0.0;
    for (uint32_t i = 0; i < count; ++i) { sum += std::pow((double)(i + 1), -(double)alpha); cdf[i] = sum; }
    for (uint32_t i = 0; i < count; ++i) cdf[i] = cdf[i] / sum;
    return cdf;
}
// Fisher-Yates with the counter-based generator
std::vector<uint32_t> seeded_permutation(uint32_t count, uint64_t base)
{
    std::vector<uint32_t> p(count);
    for (uint32_t i = 0; i < count; ++i) p[i] = i;
    for (uint32_t i = count; i-- > 1;) { const uint32_t j = (uint32_t)(mix64(base ^ (uint64_t)i) % ((uint64_t)i + 1)); std::swap(p[i], p[j]); }
    return p;
}
}  // namespace

extern "C" {

int mf_transform_float2half(const float* in, uint16_t* out, uint64_t n, void* stream)
{
    if (n == 0) return MF_OK;
    if (!in || !out) return invalid("mf_transform_float2half: null pointer");
    if ((reinterpret_cast<uintptr_t>(in) & 7) || (reinterpret_cast<uintptr_t>(out) & 3)) return invalid("mf_transform_float2half: input must be 8-byte and output 4-byte aligned");
    hipLaunchKernelGGL(float2half_kernel, dim3(stream_grid(n / 2 + 1, 4)), dim3(kStreamBlock), 0, as_stream(stream), in, out, n);
    return launch_status("mf_transform_float2half");
}
int mf_transform_half2float(const uint16_t* in, float* out, uint64_t n, void* stream)
{
    if (n == 0) return MF_OK;
    if (!in || !out) return invalid("mf_transform_half2float: null pointer");
    if ((reinterpret_cast<uintptr_t>(in) & 3) || (reinterpret_cast<uintptr_t>(out) & 7)) return invalid("mf_transform_half2float: input must be 4-byte and output 8-byte aligned");
    hipLaunchKernelGGL(half2float_kernel, dim3(stream_grid(n / 2 + 1, 4)), dim3(kStreamBlock), 0, as_stream(stream), in, out, n);
    return launch_status("mf_transform_half2float");
}

int mf_cpyparams2grouped_params(const float* original_params, void* const* converted_params,
                                const uint32_t* group_end_idx, const uint32_t* entity2group,
                                const uint32_t* entity2sorted_idx, int k, uint32_t n, uint32_t group_num, void* stream)
{
    if (k != 64 && k != 128) return invalid("mf_cpyparams2grouped_params: k must be 64 or 128 (got %d)", k);
    if (n == 0) return MF_OK;
    if (!original_params || !converted_params || !group_end_idx || !entity2group || !entity2sorted_idx || group_num == 0)
        return invalid("mf_cpyparams2grouped_params: null pointer or no groups");
    const uint32_t grid = rows_grid(n);
    if (k == 128) hipLaunchKernelGGL(scatter_to_groups_kernel<128>, dim3(grid), dim3(kBlock), 0, as_stream(stream), original_params, converted_params, group_end_idx, entity2group, entity2sorted_idx, n, group_num);
    else hipLaunchKernelGGL(scatter_to_groups_kernel<64>, dim3(grid), dim3(kBlock), 0, as_stream(stream), original_params, converted_params, group_end_idx, entity2group, entity2sorted_idx, n, group_num);
    return launch_status("mf_cpyparams2grouped_params");
}

int mf_grouped_params2dense(void* const* group_ptr, const uint32_t* group_end_idx, const uint8_t* group_prec_info,
                            float* dense, int k, uint32_t n, uint32_t group_num, void* stream)
{
    if (k != 64 && k != 128) return invalid("mf_grouped_params2dense: k must be 64 or 128 (got %d)", k);
    if (n == 0) return MF_OK;
    if (!group_ptr || !group_end_idx || !group_prec_info || !dense || group_num == 0) return invalid("mf_grouped_params2dense: null pointer or no groups");
    auto launch = [&](auto kernel, uint32_t rows) {
        hipLaunchKernelGGL(kernel, dim3(rows_grid(n, rows)), dim3(kBlock), 0, as_stream(stream), group_ptr, group_end_idx, group_prec_info, dense, n, group_num);
    };
    if (k == 64) launch(gather_from_groups_kernel<64, kRowsPerWave>, kRowsPerWave);
    else if (n <= kGatherFew) launch(gather_from_groups_kernel<128, kRowsFew>, kRowsFew);
    else launch(gather_from_groups_kernel<128, kRowsPerWave>, kRowsPerWave);
    return launch_status("mf_grouped_params2dense");
}

int mf_group_error(float* grad_sum_norm, const float* norm_sum, uint32_t norm_blocks, const uint8_t* group_prec_info,
                   const float* initial_error, float* error_out, int k, uint32_t group_num, void* stream)
{
    if (k != 64 && k != 128) return invalid("mf_group_error: k must be 64 or 128 (got %d)", k);
    if (group_num == 0) return MF_OK;
    if (!grad_sum_norm || !norm_sum || !group_prec_info || !initial_error || !error_out) return invalid("mf_group_error: null pointer");
    hipLaunchKernelGGL(group_error_kernel, dim3(group_num), dim3(kWave), 0, as_stream(stream), grad_sum_norm, norm_sum, norm_blocks, group_prec_info, initial_error, error_out, k, group_num);
    return launch_status("mf_group_error");
}

int mf_test_rmse(const mf_node* test, uint32_t test_n, const float* p, const float* q, int k, double* sum_sq, void* stream)
{
    if (k != 64 && k != 128) return invalid("mf_test_rmse: k must be 64 or 128 (got %d)", k);
    if (test_n == 0) return MF_OK;
    if (!test || !p || !q || !sum_sq) return invalid("mf_test_rmse: null pointer");
    const uint32_t grid = rmse_grid(test_n);
    if (k == 128) hipLaunchKernelGGL(rmse_dense_kernel<128>, dim3(grid), dim3(kRmseBlock), 0, as_stream(stream), test, test_n, p, q, sum_sq);
    else hipLaunchKernelGGL(rmse_dense_kernel<64>, dim3(grid), dim3(kRmseBlock), 0, as_stream(stream), test, test_n, p, q, sum_sq);
    return launch_status("mf_test_rmse");
}

int mf_test_rmse_grouped(const mf_node* test, uint32_t test_n, void* const* p, void* const* q, int k,
                         const uint32_t* user_group_end_idx, const uint32_t* item_group_end_idx,
                         const uint8_t* user_group_prec_info, const uint8_t* item_group_prec_info,
                         uint32_t user_group_num, uint32_t item_group_num, double* sum_sq, void* stream)
{
    if (k != 64 && k != 128) return invalid("mf_test_rmse_grouped: k must be 64 or 128 (got %d)", k);
    if (test_n == 0) return MF_OK;
    if (!test || !p || !q || !sum_sq || !user_group_end_idx || !item_group_end_idx || !user_group_prec_info || !item_group_prec_info)
        return invalid("mf_test_rmse_grouped: null pointer");
    if (user_group_num == 0 || item_group_num == 0) return invalid("mf_test_rmse_grouped: at least one group per side is required");
    const size_t lds = group_table_lds(user_group_num, item_group_num);
    if (lds > 60 * 1024) return invalid("mf_test_rmse_grouped: group tables need %zu bytes of LDS", lds);
    const uint32_t grid = rmse_grid(test_n);
    if (k == 128) hipLaunchKernelGGL(rmse_grouped_kernel<128>, dim3(grid), dim3(kRmseBlock), lds, as_stream(stream), test, test_n, p, q, user_group_end_idx, item_group_end_idx, user_group_prec_info, item_group_prec_info, user_group_num, item_group_num, sum_sq);
    else hipLaunchKernelGGL(rmse_grouped_kernel<64>, dim3(grid), dim3(kRmseBlock), lds, as_stream(stream), test, test_n, p, q, user_group_end_idx, item_group_end_idx, user_group_prec_info, item_group_prec_info, user_group_num, item_group_num, sum_sq);
    return launch_status("mf_test_rmse_grouped");
}

int mf_init_rand_feature(float* array, uint64_t n, uint64_t seed, uint64_t stream_id, void* stream)
{
    if (n == 0) return MF_OK;
    if (!array) return invalid("mf_init_rand_feature: null pointer");
    const uint64_t base = mix64(mix64(seed ^ 0x494E49544E4F524Dull) + stream_id);
    hipLaunchKernelGGL(init_normal_kernel, dim3(stream_grid(n)), dim3(kStreamBlock), 0, as_stream(stream), array, n, base, 0.01);
    return launch_status("mf_init_rand_feature");
}

int mf_init_idx_arr(uint32_t* arr, uint32_t n, void* stream)
{
    if (n == 0) return MF_OK;
    if (!arr) return invalid("mf_init_idx_arr: null pointer");
    hipLaunchKernelGGL(iota_kernel, dim3(stream_grid(n)), dim3(kStreamBlock), 0, as_stream(stream), arr, n);
    return launch_status("mf_init_idx_arr");
}

int mf_user_item_histogram(const mf_node* R, uint32_t n, uint32_t* user_bin, uint32_t* item_bin, void* stream)
{
    if (n == 0) return MF_OK;
    if (!R || !user_bin || !item_bin) return invalid("mf_user_item_histogram: null pointer");
    if (n <= kHistFew) {
        const uint32_t share = (n + kHistFewGrid - 1) / kHistFewGrid, per_block = share < (uint32_t)kHistBlock ? (uint32_t)kHistBlock : share;
        hipLaunchKernelGGL(histogram_few_kernel, dim3((n + per_block - 1) / per_block), dim3(kHistBlock), 0, as_stream(stream), R, n, per_block, user_bin, item_bin);
        return launch_status("mf_user_item_histogram");
    }
    if (int rc = check_hip(hipFuncSetAttribute(reinterpret_cast<const void*>(histogram_kernel), hipFuncAttributeMaxDynamicSharedMemorySize, (int)kHistLds),
                           "hipFuncSetAttribute(MaxDynamicSharedMemorySize)")) return rc;
    hipLaunchKernelGGL(histogram_kernel, dim3(kHistGrid), dim3(kHistBlock), kHistLds, as_stream(stream), R, n, user_bin, item_bin);
    return launch_status("mf_user_item_histogram");
}

int mf_matrix_reconst_triplet(mf_node* R, const uint32_t* user2sorted_idx, const uint32_t* item2sorted_idx, uint32_t n, void* stream)
{
    if (n == 0) return MF_OK;
    if (!R || !user2sorted_idx || !item2sorted_idx) return invalid("mf_matrix_reconst_triplet: null pointer");
    const uint64_t words = (uint64_t)n * 3;
    auto launch = [&](auto kernel, int unroll) {
        hipLaunchKernelGGL(kernel, dim3(stream_grid(words / 4 + 1, unroll)), dim3(kStreamBlock), 0, as_stream(stream), reinterpret_cast<uint32_t*>(R), user2sorted_idx, item2sorted_idx, words);
    };
    if (words / 4 <= 3u << 18) launch(reindex_kernel<1>, 1);
    else launch(reindex_kernel<4>, 4);
    return launch_status("mf_matrix_reconst_triplet");
}

int mf_row_traffic_probe(const mf_node* R, uint32_t n, void* p, void* q, uint32_t row_bytes, uint32_t num_workers,
                         uint64_t seed, void* stream, const mf_hogwild_options* options)
{
    return mf_row_traffic_probe_sides(R, n, p, q, row_bytes, row_bytes, num_workers, seed, stream, options);
}
int mf_row_traffic_probe_sides(const mf_node* R, uint32_t n, void* p, void* q, uint32_t row_bytes, uint32_t item_row_bytes, uint32_t num_workers,
                               uint64_t seed, void* stream, const mf_hogwild_options* options)
{
    if (n == 0) return MF_OK;
    if (!R || !p || !q) return invalid("mf_row_traffic_probe: null pointer");
    if (row_bytes != 128 && row_bytes != 256 && row_bytes != 512) return invalid("mf_row_traffic_probe: row_bytes must be 128, 256 or 512 (got %u)", row_bytes);
    if (item_row_bytes != 128 && item_row_bytes != 256 && item_row_bytes != 512) return invalid("mf_row_traffic_probe: row_bytes must be 128, 256 or 512 (got %u)", item_row_bytes);
    if (num_workers == 0) return invalid("mf_row_traffic_probe: num_workers must be positive");
    mf_hogwild_options o = {};
    if (options) o = *options;
    if ((o.user_keep == nullptr) != (o.item_keep == nullptr)) return invalid("mf_row_traffic_probe: give both keep tables or neither");
    if ((o.user_slots && (!o.user_slot || !o.user_replicas)) || (o.item_slots && (!o.item_slot || !o.item_replicas))) return invalid("mf_row_traffic_probe: replicated rows need slot tables and replica arrays");
    if ((reinterpret_cast<uintptr_t>(p) | reinterpret_cast<uintptr_t>(q)) & 7) return invalid("mf_row_traffic_probe: rows must be 8-byte aligned");
    const bool coherent = o.cached_rows == 0;
    const uint8_t* user_keep = o.user_keep; const uint8_t* item_keep = o.item_keep;
    const uint32_t per_worker = (uint32_t)(((uint64_t)n + num_workers - 1) / num_workers);
    const dim3 grid((num_workers + kWavesPerBlock - 1) / kWavesPerBlock), block(kBlock);
    uint8_t* P = static_cast<uint8_t*>(p); uint8_t* Q = static_cast<uint8_t*>(q);
    uint8_t* RP = static_cast<uint8_t*>(o.user_replicas); uint8_t* RQ = static_cast<uint8_t*>(o.item_replicas);
    const uint64_t key = mix64(seed ^ 0x70726f6265ull);
#define MF_PROBE(BYTES, COH) hipLaunchKernelGGL((row_traffic_probe_kernel<BYTES, COH>), grid, block, 0, as_stream(stream), R, n, P, Q, per_worker, user_keep, item_keep, o.user_slot, o.item_slot, o.user_slots, o.item_slots, RP, RQ, key, 0u)
#define MF_PROBE2(BP, BQ) hipLaunchKernelGGL((row_traffic_probe_kernel<BP, true, BQ>), grid, block, 0, as_stream(stream), R, n, P, Q, per_worker, user_keep, item_keep, o.user_slot, o.item_slot, o.user_slots, o.item_slots, RP, RQ, key, 0u)
    if (row_bytes != item_row_bytes) {
        // rows of different widths on the two sides: MASCOT after one side's groups have been promoted
        if (!coherent) return invalid("mf_row_traffic_probe_sides: sides of different widths are probed with device-coherent stores only");
        if (row_bytes == 256 && item_row_bytes == 512) MF_PROBE2(4, 8);
        else if (row_bytes == 512 && item_row_bytes == 256) MF_PROBE2(8, 4);
        else if (row_bytes == 128 && item_row_bytes == 256) MF_PROBE2(2, 4);
        else if (row_bytes == 256 && item_row_bytes == 128) MF_PROBE2(4, 2);
        else return invalid("mf_row_traffic_probe_sides: the wider side's rows must be twice the other's");
    }
    else if (row_bytes == 128) { if (coherent) MF_PROBE(2, true); else MF_PROBE(2, false); }
    else if (row_bytes == 256) { if (coherent) MF_PROBE(4, true); else MF_PROBE(4, false); }
    else { if (coherent) MF_PROBE(8, true); else MF_PROBE(8, false); }
#undef MF_PROBE2
#undef MF_PROBE
    return launch_status("mf_row_traffic_probe");
}

int mf_synth_baseline_config(int config, mf_synth_config* out)
{
    if (!out) return invalid("mf_synth_baseline_config: null pointer");
    //                          users    items    train       test     alpha_u alpha_i rank noise  mean  step  lo    hi   bimodal
    static const mf_synth_config table[5] = {
        {5000u, 2000u, 400000ull, 100000ull, 1.0f, 1.0f, 8u, 0.8f, 3.5f, 1.0f, 1.0f, 5.0f, 0u},
        {70000u, 10700u, 8000000ull, 2000000ull, 0.9f, 0.9f, 16u, 0.8f, 3.5f, 0.5f, 0.5f, 5.0f, 0u},
        {162000u, 59000u, 20000000ull, 5000000ull, 1.0f, 1.0f, 16u, 0.8f, 3.5f, 0.5f, 0.5f, 5.0f, 0u},
        {480000u, 17800u, 100000000ull, 1400000ull, 0.8f, 1.1f, 32u, 0.9f, 3.6f, 1.0f, 1.0f, 5.0f, 0u},
        {1000000u, 625000u, 250000000ull, 4000000ull, 1.2f, 1.2f, 0u, 15.0f, 0.0f, 1.0f, 0.0f, 100.0f, 1u},
    };
    if (config < 1 || config > 5) return invalid("mf_synth_baseline_config: configurations are numbered 1..5 (got %d)", config);
    *out = table[config - 1];
    return MF_OK;
}

static int check_synth(const char* who, const mf_synth_config* cfg)
{
    if (!cfg) return invalid("%s: null configuration", who);
    if (cfg->n_users == 0 || cfg->n_items == 0) return invalid("%s: no users or no items", who);
    if (!cfg->bimodal && (cfg->rank == 0 || cfg->rank > 1024u)) return invalid("%s: rank must be 1..1024 (got %u)", who, cfg->rank);
    if (!(cfg->step > 0.0f) || !(cfg->lo <= cfg->hi)) return invalid("%s: step must be positive and lo <= hi", who);
    return MF_OK;
}
// Workspace layout of the generator's tables: user CDF, item CDF (binary64), user permutation, item permutation
// (uint32), and unless bimodal the factors U [users][rank], V [items][rank] (binary32); every part 256-byte aligned.
struct SynthLayout { size_t ucdf, icdf, uperm, iperm, U, V, total; };
static SynthLayout synth_layout(const mf_synth_config& c)
{
    auto al = [](size_t b) { return (b + 255) / 256 * 256; };
    SynthLayout l;
    l.ucdf = 0; l.icdf = l.ucdf + al((size_t)c.n_users * 8); l.uperm = l.icdf + al((size_t)c.n_items * 8);
    l.iperm = l.uperm + al((size_t)c.n_users * 4); l.U = l.iperm + al((size_t)c.n_items * 4);
    const size_t fu = c.bimodal ? 0 : al((size_t)c.n_users * c.rank * 4), fv = c.bimodal ? 0 : al((size_t)c.n_items * c.rank * 4);
    l.V = l.U + fu; l.total = l.V + fv;
    return l;
}
static SynthTables synth_tables(const mf_synth_config& c, const void* workspace)
{
    const SynthLayout l = synth_layout(c);
    const uint8_t* ws = static_cast<const uint8_t*>(workspace);
    SynthTables t = {};
    t.user_cdf = reinterpret_cast<const double*>(ws + l.ucdf); t.item_cdf = reinterpret_cast<const double*>(ws + l.icdf);
    t.user_perm = reinterpret_cast<const uint32_t*>(ws + l.uperm); t.item_perm = reinterpret_cast<const uint32_t*>(ws + l.iperm);
    if (!c.bimodal) { t.U = reinterpret_cast<const float*>(ws + l.U); t.V = reinterpret_cast<const float*>(ws + l.V); }
    return t;
}
static uint64_t synth_key(uint64_t seed) { return mix64(seed ^ 0x53594E5448455449ull); }

size_t mf_synth_tables_bytes(const mf_synth_config* cfg)
{
    if (check_synth("mf_synth_tables_bytes", cfg)) return 0;
    return synth_layout(*cfg).total;
}
int mf_synth_build_tables(const mf_synth_config* cfg, uint64_t seed, void* workspace, size_t workspace_bytes, void* stream)
{
    if (int rc = check_synth("mf_synth_build_tables", cfg)) return rc;
    const mf_synth_config c = *cfg;
    const SynthLayout l = synth_layout(c);
    if (!workspace || reinterpret_cast<uintptr_t>(workspace) % 256) return invalid("mf_synth_build_tables: the workspace must be non-null and 256-byte aligned");
    if (workspace_bytes < l.total) return invalid("mf_synth_build_tables: the workspace holds %zu bytes, the tables need %zu (mf_synth_tables_bytes)", workspace_bytes, l.total);
    hipStream_t st = as_stream(stream);
    uint8_t* ws = static_cast<uint8_t*>(workspace);
    const uint64_t key = synth_key(seed);
    const std::vector<double> ucdf = zipf_cdf(c.n_users, c.user_alpha), icdf = zipf_cdf(c.n_items, c.item_alpha);
    const std::vector<uint32_t> uperm = seeded_permutation(c.n_users, mix64(key + 1)), iperm = seeded_permutation(c.n_items, mix64(key + 2));
    if (int rc = check_hip(hipMemcpyAsync(ws + l.ucdf, ucdf.data(), ucdf.size() * 8, hipMemcpyHostToDevice, st), "hipMemcpyAsync(synthetic tables)")) return rc;
    if (int rc = check_hip(hipMemcpyAsync(ws + l.icdf, icdf.data(), icdf.size() * 8, hipMemcpyHostToDevice, st), "hipMemcpyAsync(synthetic tables)")) return rc;
    if (int rc = check_hip(hipMemcpyAsync(ws + l.uperm, uperm.data(), uperm.size() * 4, hipMemcpyHostToDevice, st), "hipMemcpyAsync(synthetic tables)")) return rc;
    if (int rc = check_hip(hipMemcpyAsync(ws + l.iperm, iperm.data(), iperm.size() * 4, hipMemcpyHostToDevice, st), "hipMemcpyAsync(synthetic tables)")) return rc;
    if (!c.bimodal) {
        const uint64_t nu = (uint64_t)c.n_users * c.rank, nv = (uint64_t)c.n_items * c.rank;
        hipLaunchKernelGGL(init_normal_kernel, dim3(stream_grid(nu)), dim3(kStreamBlock), 0, st, reinterpret_cast<float*>(ws + l.U), nu, mix64(key + 3), 0.5);
        hipLaunchKernelGGL(init_normal_kernel, dim3(stream_grid(nv)), dim3(kStreamBlock), 0, st, reinterpret_cast<float*>(ws + l.V), nv, mix64(key + 4), 0.5);
        if (int rc = launch_status("mf_synth_build_tables")) return rc;
    }
    // the host-side tables above go out of scope on return: wait for their copies (the one synchronisation of the generator)
    return check_hip(hipStreamSynchronize(st), "mf_synth_build_tables: hipStreamSynchronize");
}
int mf_generate_ratings_ws(const mf_synth_config* cfg, uint64_t seed, const void* tables, uint64_t first, uint64_t count, mf_node* out, void* stream)
{
    if (int rc = check_synth("mf_generate_ratings_ws", cfg)) return rc;
    if (count == 0) return MF_OK;
    if (!out || !tables) return invalid("mf_generate_ratings_ws: null output or tables");
    const mf_synth_config c = *cfg;
    hipLaunchKernelGGL(generate_ratings_kernel, dim3(stream_grid(count)), dim3(kStreamBlock), 0, as_stream(stream), c, synth_tables(c, tables), synth_key(seed), first, count, 1.0f / c.step, out);
    return launch_status("mf_generate_ratings_ws");
}
int mf_generate_ratings(const mf_synth_config* cfg, uint64_t seed, uint64_t first, uint64_t count, mf_node* out, void* stream)
{
    if (int rc = check_synth("mf_generate_ratings", cfg)) return rc;
    if (count == 0) return MF_OK;
    if (!out) return invalid("mf_generate_ratings: null output");
    const size_t bytes = synth_layout(*cfg).total;
    void* ws = nullptr;
    if (int rc = check_hip(hipMalloc(&ws, bytes), "mf_generate_ratings: hipMalloc(tables)")) return rc;
    int rc = mf_synth_build_tables(cfg, seed, ws, bytes, stream);
    if (rc == MF_OK) rc = mf_generate_ratings_ws(cfg, seed, ws, first, count, out, stream);
    if (rc == MF_OK) rc = check_hip(hipStreamSynchronize(as_stream(stream)), "mf_generate_ratings: hipStreamSynchronize");       // the tables are freed on return
    (void)hipFree(ws);
    return rc;
}

int mf_generate_ratings_host(const mf_synth_config* cfg, uint64_t seed, uint64_t first, uint64_t count, mf_node* host_out)
{
    if (count == 0) return MF_OK;
    if (!host_out) return invalid("mf_generate_ratings_host: null output");
    void* dev = nullptr;
    if (int rc = check_hip(hipMalloc(&dev, count * sizeof(mf_node)), "mf_generate_ratings_host: hipMalloc")) return rc;
    int rc = mf_generate_ratings(cfg, seed, first, count, static_cast<mf_node*>(dev), nullptr);
    if (rc == MF_OK) rc = check_hip(hipMemcpy(host_out, dev, count * sizeof(mf_node), hipMemcpyDeviceToHost), "mf_generate_ratings_host: hipMemcpy");
    (void)hipFree(dev);
    return rc;
}

}  // extern "C"
