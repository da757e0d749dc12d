// Popularity sort (thrust::sort_by_key in the reference, preprocess_utils.h:87-88; a rocPRIM stable LSD radix sort) and
// the seeded rating shuffle (std::random_shuffle, mf_methods.cu:38-39) on the device.
#include "mf_host.h"
#include "mf_device.h"
#include <cstring>
#include <mutex>
#include <type_traits>
#include <rocprim/device/device_radix_sort.hpp>

namespace mf {

// ---- shuffle: ratings in ascending order of the 64-bit key mix64(base ^ position) ------------------------------------
// The keys are a bijection of the positions, so they are all different (the order is unique, and nothing has to be stable)
// and a key never has to be stored: 4 bytes of position stand for it.  They are also spread evenly, so their leading bits
// cut the ratings into buckets of nearly equal size, small enough to be put in order inside one workgroup's LDS:
//   count     ratings per leading digit and workgroup: arithmetic only, nothing is read
//   partition one pass (up to kOneLevelBits leading bits) or two: tiles of kTile ratings are grouped by digit in LDS and
//             written in runs; what moves is the rating itself and its position, 16 bytes
//   finish    one workgroup per bucket: ordered by the next 12 bits of the key, ties by the whole key, written in order
// What bounds it is memory traffic: 16 bytes written, read and written again, read, and 12 bytes written.  A radix sort of
// (key, position) pairs moved 24 bytes eight times and then gathered the ratings from random places, a cache line for
// each 12 bytes: at 100M ratings 9.7 ms, of which the gather took 2.7; this takes 2.6 (the two partition passes 0.76 and 0.75,
// at 3.7 and 4.3 TB/s, the counts 0.45, the finish 0.65).  Rating and position move as one 16-byte record: in two arrays the
// partition passes took 0.88 each, a lane's two stores ending in twice as many partly written lines (the second count, which
// reads positions alone, 0.1 less).
constexpr int kShufBlock = 512;                   // the placing and the finishing kernel
constexpr uint32_t kPerThread = 8;
constexpr uint32_t kBucketCap = kShufBlock * kPerThread;      // ratings that the finishing workgroup orders in LDS
// The buckets are cut for at most this many ratings on average; the keys being spread evenly, kBucketCap lies 18 standard
// deviations above it (and a larger bucket is only slow).
constexpr uint32_t kBucketMean = 3072;
// Up to 256 buckets one pass leaves runs of at least 16 ratings per tile and digit (256 bytes); from there on two passes of
// half the bits each are cheaper than one with shorter runs.
constexpr int kOneLevelBits = 8;
constexpr uint32_t kSubBits = 12, kSubBins = 1u << kSubBits;
struct Node3 { uint32_t r, u, i; };               // an mf_node as its three words
static_assert(sizeof(Node3) == sizeof(mf_node), "a rating is three words");

// digit of `bits` bits that follows the first `skip` bits of a key (bits >= 1)
__device__ __forceinline__ uint32_t key_digit(uint64_t key, int skip, int bits) { return (uint32_t)((key << skip) >> (64 - bits)); }

// Exclusive scan of v[0..bins) in place by one workgroup of BLOCK threads.  part: one word per wavefront.
template <int BLOCK> __device__ __forceinline__ void block_scan(uint32_t* v, uint32_t bins, uint32_t* part)
{
    const uint32_t per = (bins + BLOCK - 1) / BLOCK, first = threadIdx.x * per;
    uint32_t sum = 0;
    for (uint32_t i = 0; i < per; ++i) if (first + i < bins) sum += v[first + i];
    uint32_t incl = sum;
    for (int d = 1; d < kWave; d <<= 1) { const uint32_t o = __shfl_up(incl, d); if ((int)(threadIdx.x & 63) >= d) incl += o; }
    if ((threadIdx.x & 63) == 63) part[threadIdx.x >> 6] = incl;
    __syncthreads();
    uint32_t before = 0;
    for (uint32_t w = 0; w < (threadIdx.x >> 6); ++w) before += part[w];
    uint32_t at = before + incl - sum;
    for (uint32_t i = 0; i < per; ++i) if (first + i < bins) { const uint32_t c = v[first + i]; v[first + i] = at; at += c; }
    __syncthreads();
}

// A rating and its position, where they have been moved together, or from the original order.  Which it is is known at compile
// time: with a branch between them every load would be waited for before the next.
template <bool MOVED> __device__ __forceinline__ uint4 record(const uint4* moved, const Node3* nodes, uint32_t at)
{
    if constexpr (MOVED) return moved[at];
    const Node3 x = nodes[at];
    return make_uint4(x.r, x.u, x.i, at);
}

// What a workgroup of a pass works on: ratings [begin, end) of the input, which all belong to segment `seg` (one segment,
// the whole input, in the first pass; the first pass's buckets in the second), as chunk `chunk` of that segment.
struct PassArgs {
    const Node3* nodes;           // the first pass's input
    const uint4* moved;           // the second's: a rating and its position; null in the first pass
    uint4* moved_out;
    uint32_t n; uint64_t base;
    int skip, bits;               // the digit of this pass
    uint32_t chunks;              // workgroups per segment
    const uint32_t* seg_start;    // null: one segment
    uint32_t segs;
    uint32_t* table;              // [seg][chunk][digit] counts, then starting places (place_kernel)
    uint32_t* bucket_start;       // [seg][digit]
};
template <uint32_t TILE> __device__ __forceinline__ void chunk_of(const PassArgs& a, uint32_t& seg, uint32_t& begin, uint32_t& end)
{
    seg = blockIdx.x / a.chunks;
    const uint32_t chunk = blockIdx.x % a.chunks;
    const uint32_t s0 = a.seg_start ? a.seg_start[seg] : 0u, s1 = a.seg_start && seg + 1 < a.segs ? a.seg_start[seg + 1] : a.n;
    const uint32_t tiles = (uint32_t)(((uint64_t)(s1 - s0) + TILE - 1) / TILE), per = (tiles + a.chunks - 1) / a.chunks;
    const uint64_t b = (uint64_t)s0 + (uint64_t)per * TILE * chunk, e = b + (uint64_t)per * TILE;
    begin = b < s1 ? (uint32_t)b : s1; end = e < s1 ? (uint32_t)e : s1;
}
template <int BLOCK> __global__ __launch_bounds__(BLOCK) void shuffle_count_kernel(PassArgs a)
{
    extern __shared__ uint32_t shuf_smem[];
    uint32_t* cnt = shuf_smem;
    const uint32_t bins = 1u << a.bits;
    for (uint32_t d = threadIdx.x; d < bins; d += BLOCK) cnt[d] = 0u;
    __syncthreads();
    uint32_t seg, begin, end;
    chunk_of<BLOCK * kPerThread>(a, seg, begin, end);
#pragma unroll 4
    for (uint64_t i = (uint64_t)begin + threadIdx.x; i < end; i += BLOCK) {
        const uint32_t pos = a.moved ? a.moved[i].w : (uint32_t)i;
        atomicAdd(&cnt[key_digit(mix64(a.base ^ (uint64_t)pos), a.skip, a.bits)], 1u);
    }
    __syncthreads();
    for (uint32_t d = threadIdx.x; d < bins; d += BLOCK) a.table[(size_t)blockIdx.x * bins + d] = cnt[d];
}
// counts -> the place where each workgroup's ratings of each digit begin; one workgroup per segment
__global__ __launch_bounds__(kShufBlock) void shuffle_place_kernel(PassArgs a)
{
    extern __shared__ uint32_t shuf_smem[];
    uint32_t* first = shuf_smem;
    __shared__ uint32_t part[kShufBlock / kWave];
    const uint32_t bins = 1u << a.bits, seg = blockIdx.x;
    uint32_t* t = a.table + (size_t)seg * a.chunks * bins;
    // digits across the lanes, and the chunks split over as many groups of lanes as there are digits to spare
    const uint32_t groups = bins < (uint32_t)kShufBlock ? kShufBlock / bins : 1u, per = (a.chunks + groups - 1) / groups;
    uint32_t* sums = first + bins;      // [groups][bins]
    const uint32_t g = bins < (uint32_t)kShufBlock ? threadIdx.x / bins : 0u;
    const uint32_t step = bins < (uint32_t)kShufBlock ? bins : (uint32_t)kShufBlock;
    const uint32_t c0 = g * per < a.chunks ? g * per : a.chunks, c1 = c0 + per < a.chunks ? c0 + per : a.chunks;
    for (uint32_t d = threadIdx.x % step; d < bins; d += step) {
        uint32_t s = 0;
#pragma unroll 16
        for (uint32_t c = c0; c < c1; ++c) s += t[(size_t)c * bins + d];
        sums[(size_t)g * bins + d] = s;
    }
    __syncthreads();
    for (uint32_t d = threadIdx.x; d < bins; d += kShufBlock) {
        uint32_t s = 0;
        for (uint32_t h = 0; h < groups; ++h) { const uint32_t v = sums[(size_t)h * bins + d]; sums[(size_t)h * bins + d] = s; s += v; }
        first[d] = s;
    }
    __syncthreads();
    block_scan<kShufBlock>(first, bins, part);
    const uint32_t s0 = a.seg_start ? a.seg_start[seg] : 0u;
    for (uint32_t d = threadIdx.x; d < bins; d += kShufBlock) a.bucket_start[(size_t)seg * bins + d] = s0 + first[d];
    for (uint32_t d = threadIdx.x % step; d < bins; d += step) {
        uint32_t at = s0 + first[d] + sums[(size_t)g * bins + d];
        uint32_t c = c0;
        for (; c + 16 <= c1; c += 16) {        // sixteen loads in flight
            uint32_t v[16];
#pragma unroll
            for (int j = 0; j < 16; ++j) v[j] = t[(size_t)(c + j) * bins + d];
#pragma unroll
            for (int j = 0; j < 16; ++j) { t[(size_t)(c + j) * bins + d] = at; at += v[j]; }
        }
        for (; c < c1; ++c) { const uint32_t v = t[(size_t)c * bins + d]; t[(size_t)c * bins + d] = at; at += v; }
    }
}
static size_t place_lds(int bits) { const size_t bins = (size_t)1 << bits; return (bins + (bins < (size_t)kShufBlock ? (size_t)kShufBlock : bins)) * 4; }

// Each lane has 8 ratings in flight.  Up to 256 digits one workgroup of 1024 threads (147 KB of LDS) on a compute unit, two of 512 up
// to 512 digits (76 KB each), one of 512 from there on (from 805M ratings).  The larger tile writes runs twice as long, and with half as many
// workgroups the cache lines that are partly written at any time fit in an XCD's L2.
template <int BLOCK, bool MOVED> __global__ __launch_bounds__(BLOCK) void shuffle_partition_kernel(PassArgs a)
{
    constexpr uint32_t kTile = BLOCK * kPerThread;
    extern __shared__ __align__(16) uint32_t shuf_smem[];
    __shared__ uint32_t part[BLOCK / kWave];
    const uint32_t bins = 1u << a.bits;
    uint4* stage = reinterpret_cast<uint4*>(shuf_smem);                         // kTile ratings, grouped by digit
    uint32_t* cnt = shuf_smem + kTile * 4;                                      // ratings per digit, then where they begin in `stage`
    uint32_t* next = cnt + bins;                                                // where this workgroup's next rating of a digit goes
    uint16_t* digit_of = reinterpret_cast<uint16_t*>(next + bins);              // digit of a staged rating
    for (uint32_t d = threadIdx.x; d < bins; d += BLOCK) next[d] = a.table[(size_t)blockIdx.x * bins + d];
    uint32_t seg, begin, end;
    chunk_of<kTile>(a, seg, begin, end);
    uint4 rec[kPerThread];
    auto fetch = [&](uint64_t tile) {      // without a branch per load, which would be waited for; past the end the last rating again
        if (tile >= end) return;
        const uint32_t most = end - tile < kTile ? (uint32_t)(end - tile) - 1u : kTile - 1u;
#pragma unroll
        for (uint32_t j = 0; j < kPerThread; ++j) rec[j] = record<MOVED>(a.moved, a.nodes, (uint32_t)tile + min(j * BLOCK + threadIdx.x, most));
    };
    fetch(begin);
    for (uint64_t tile = begin; tile < end; tile += kTile) {
        const uint32_t m = end - tile < kTile ? (uint32_t)(end - tile) : kTile;
        for (uint32_t d = threadIdx.x; d < bins; d += BLOCK) cnt[d] = 0u;
        __syncthreads();
        uint32_t digit[kPerThread], rank[kPerThread];
#pragma unroll
        for (uint32_t j = 0; j < kPerThread; ++j) {
            if (j * BLOCK + threadIdx.x < m) {
                digit[j] = key_digit(mix64(a.base ^ (uint64_t)rec[j].w), a.skip, a.bits);
                rank[j] = atomicAdd(&cnt[digit[j]], 1u);
            }
        }
        __syncthreads();
        block_scan<BLOCK>(cnt, bins, part);
#pragma unroll
        for (uint32_t j = 0; j < kPerThread; ++j) {
            if (j * BLOCK + threadIdx.x < m) {
                const uint32_t at = cnt[digit[j]] + rank[j];
                stage[at] = rec[j];
                digit_of[at] = (uint16_t)digit[j];
            }
        }
        __syncthreads();
        fetch(tile + kTile);        // on their way while this tile is written
#pragma unroll
        for (uint32_t j = 0; j < kPerThread; ++j) {
            const uint32_t o = j * BLOCK + threadIdx.x;
            if (o < m) {
                const uint32_t d = digit_of[o];
                a.moved_out[next[d] + (o - cnt[d])] = stage[o];
            }
        }
        __syncthreads();
        for (uint32_t d = threadIdx.x; d < bins; d += BLOCK) next[d] += (d + 1 < bins ? cnt[d + 1] : m) - cnt[d];
        __syncthreads();
    }
}
constexpr int kLargeTileBits = 8;
static size_t partition_lds(int bits) { const size_t tile = (bits <= kLargeTileBits ? 1024u : 512u) * kPerThread; return tile * 18 + ((size_t)8 << bits); }
// of the kernel on the whole card: 256 compute units of 160 KB
static uint32_t partition_resident(int bits) { return 256u * (uint32_t)((160u << 10) / (partition_lds(bits) + 1024 / kWave * 4)); }

// One bucket in order: by the kSubBits bits of the key after the bucket's, in LDS (0.75 ratings per value on average), then by
// the whole key among the ratings that share them.  64 KB of LDS: two workgroups per compute unit.
template <bool MOVED>
__global__ __launch_bounds__(kShufBlock) void shuffle_finish_kernel(const uint4* __restrict__ moved, const Node3* __restrict__ nodes, Node3* __restrict__ out,
                                                                    uint32_t n, uint64_t base, int skip, const uint32_t* __restrict__ bucket_start, uint32_t buckets)
{
    __shared__ uint32_t first[kSubBins];
    __shared__ __align__(16) uint32_t stage[kBucketCap * 3];      // keys, then ratings
    __shared__ uint32_t part[kShufBlock / kWave];
    const uint32_t begin = bucket_start ? bucket_start[blockIdx.x] : 0u, end = bucket_start && blockIdx.x + 1 < buckets ? bucket_start[blockIdx.x + 1] : n;
    const uint32_t m = end - begin;
    if (m > kBucketCap) {       // larger than the LDS: each rating's place is counted out
        for (uint32_t o = threadIdx.x; o < m; o += kShufBlock) {
            const uint4 x = record<MOVED>(moved, nodes, begin + o);
            const uint64_t key = mix64(base ^ (uint64_t)x.w);
            uint32_t rank = 0;
            for (uint32_t q = 0; q < m; ++q) rank += mix64(base ^ (uint64_t)record<MOVED>(moved, nodes, begin + q).w) < key ? 1u : 0u;
            out[begin + rank] = Node3{x.x, x.y, x.z};
        }
        return;
    }
    if (m == 0u) return;
    for (uint32_t d = threadIdx.x; d < kSubBins; d += kShufBlock) first[d] = 0u;
    uint4 rec[kPerThread]; uint64_t key[kPerThread]; uint32_t place[kPerThread];
#pragma unroll
    for (uint32_t j = 0; j < kPerThread; ++j) rec[j] = record<MOVED>(moved, nodes, begin + min(j * kShufBlock + threadIdx.x, m - 1u));
    __syncthreads();
#pragma unroll
    for (uint32_t j = 0; j < kPerThread; ++j) {
        if (j * kShufBlock + threadIdx.x < m) {
            key[j] = mix64(base ^ (uint64_t)rec[j].w);
            place[j] = atomicAdd(&first[key_digit(key[j], skip, kSubBits)], 1u);
        }
    }
    __syncthreads();
    block_scan<kShufBlock>(first, kSubBins, part);
    uint64_t* keys = reinterpret_cast<uint64_t*>(stage);
#pragma unroll
    for (uint32_t j = 0; j < kPerThread; ++j)
        if (j * kShufBlock + threadIdx.x < m) keys[first[key_digit(key[j], skip, kSubBits)] + place[j]] = key[j];
    __syncthreads();
#pragma unroll
    for (uint32_t j = 0; j < kPerThread; ++j) {
        if (j * kShufBlock + threadIdx.x < m) {
            const uint32_t d = key_digit(key[j], skip, kSubBits), b = first[d], e = d + 1 < kSubBins ? first[d + 1] : m;
            uint32_t at = b;
            for (uint32_t q = b; q < e; ++q) at += keys[q] < key[j] ? 1u : 0u;
            place[j] = at;
        }
    }
    __syncthreads();
#pragma unroll
    for (uint32_t j = 0; j < kPerThread; ++j)
        if (j * kShufBlock + threadIdx.x < m) { stage[place[j] * 3] = rec[j].x; stage[place[j] * 3 + 1] = rec[j].y; stage[place[j] * 3 + 2] = rec[j].z; }
    __syncthreads();
    uint32_t* to = reinterpret_cast<uint32_t*>(out + begin);
    for (uint32_t w = threadIdx.x; w < m * 3; w += kShufBlock) to[w] = stage[w];
}

struct DeviceBuffers {
    void* ptr[4] = {nullptr, nullptr, nullptr, nullptr};
    ~DeviceBuffers() { for (void* p : ptr) if (p) (void)hipFree(p); }
};

constexpr size_t kAlign = 256;
static inline size_t aligned(size_t bytes) { return (bytes + kAlign - 1) / kAlign * kAlign; }

// Workspace layout of the count sort: sorted counts, sorted ids (the radix sort's output buffers), rocPRIM's own
// temporary storage.  The size query only computes sizes; it needs a current device (rocPRIM picks its kernel
// configuration by architecture).
static int sort_layout(uint32_t n, size_t* tmp_bytes, size_t* total)
{
    size_t tmp = 0;
    uint32_t* none = nullptr;
    if (int rc = check_hip(rocprim::radix_sort_pairs(nullptr, tmp, none, none, none, none, (size_t)n, 0, 32, nullptr), "radix_sort_pairs(size)")) return rc;
    *tmp_bytes = tmp;
    *total = 2 * aligned((size_t)n * 4) + aligned(tmp ? tmp : 4);
    return MF_OK;
}
static int sort_in(uint32_t* cnt, uint32_t* idx, uint32_t n, uint8_t* ws, size_t tmp_bytes, hipStream_t s)
{
    uint32_t* cnt_out = reinterpret_cast<uint32_t*>(ws);
    uint32_t* idx_out = reinterpret_cast<uint32_t*>(ws + aligned((size_t)n * 4));
    void* tmp = ws + 2 * aligned((size_t)n * 4);
    if (int rc = check_hip(rocprim::radix_sort_pairs(tmp, tmp_bytes, cnt, cnt_out, idx, idx_out, (size_t)n, 0, 32, s), "mf_sort_by_count: radix_sort_pairs")) return rc;
    if (int rc = check_hip(hipMemcpyAsync(cnt, cnt_out, (size_t)n * 4, hipMemcpyDeviceToDevice, s), "mf_sort_by_count: copy")) return rc;
    return check_hip(hipMemcpyAsync(idx, idx_out, (size_t)n * 4, hipMemcpyDeviceToDevice, s), "mf_sort_by_count: copy");
}
// The shuffle's passes and its workspace: positions and ratings after the first and after the second pass, the table of
// counts of each pass and the beginnings of the buckets.
struct ShufflePlan {
    int bits1 = 0, bits2 = 0;
    uint32_t chunks1 = 0, chunks2 = 0;
    size_t moved[2], table[2], start[2], total = 0;
};
static ShufflePlan shuffle_plan(uint32_t n)
{
    ShufflePlan p;
    int bits = 0;
    while (((uint64_t)n + (1ull << bits) - 1) >> bits > kBucketMean) ++bits;
    p.bits1 = bits <= kOneLevelBits ? bits : (bits + 1) / 2;
    p.bits2 = bits - p.bits1;
    // as many workgroups as are resident, and at least four tiles for each where the input has them
    auto chunks = [](int b, uint64_t ratings, uint32_t segs) {
        const uint64_t tile = (b <= kLargeTileBits ? 1024u : 512u) * kPerThread, by_size = (ratings + 4 * tile - 1) / (4 * tile);
        const uint32_t most = partition_resident(b) / segs;
        return by_size < 1 || most < 1 ? 1u : (by_size < most ? (uint32_t)by_size : most);
    };
    p.chunks1 = chunks(p.bits1, n, 1);
    p.chunks2 = chunks(p.bits2, (uint64_t)n >> p.bits1, 1u << p.bits1);
    auto take = [&](size_t bytes) { const size_t at = p.total; p.total += aligned(bytes); return at; };
    for (int l = 0; l < 2; ++l) {
        const int b = l ? p.bits2 : p.bits1;
        if (!b) continue;
        p.moved[l] = take((size_t)n * sizeof(uint4));
        p.table[l] = take(l ? (((size_t)p.chunks2 << p.bits1) << p.bits2) * 4 : ((size_t)p.chunks1 << p.bits1) * 4);
        p.start[l] = take(((size_t)1 << (l ? p.bits1 + p.bits2 : p.bits1)) * 4);
    }
    if (p.total == 0) p.total = kAlign;
    return p;
}

// ---- scratch of mf_sort_by_count_static ------------------------------------------------------------------------
// Device memory that belongs to the library image: every GPU the library runs on holds its own copy from the moment
// the code object is loaded until the process ends.  20 MiB: the two output buffers of a sort of kStaticSortMax
// counts (8 MiB) and rocPRIM's temporary storage for that size (8.4 MB on gfx950 with rocPRIM 4: its own pair of
// buffers and its counters).
constexpr uint32_t kStaticSortMax = 1u << 20;
constexpr size_t kStaticScratchBytes = 20u << 20;
static __device__ __align__(256) unsigned char scratch[kStaticScratchBytes];
// The array's name is a host-side stand-in, not a device address: the address of each device's copy is asked for once,
// with that device current, and everything below uses that pointer.
constexpr int kMaxDevices = 64;
static std::mutex g_scratch_mutex;
static void* g_scratch_ptr[kMaxDevices] = {};
static int static_scratch(void** out)
{
    int dev = 0;
    if (int rc = check_hip(hipGetDevice(&dev), "mf_sort_by_count_static: hipGetDevice")) return rc;
    if (dev < 0 || dev >= kMaxDevices) return invalid("mf_sort_by_count_static: device %d is beyond the %d devices this library keeps scratch addresses for", dev, kMaxDevices);
    std::lock_guard<std::mutex> lock(g_scratch_mutex);
    if (!g_scratch_ptr[dev]) {
        void* ptr = nullptr;
        if (int rc = check_hip(hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)), "mf_sort_by_count_static: hipGetSymbolAddress(scratch)")) return rc;
        if (!ptr) return invalid("mf_sort_by_count_static: the scratch array has no address on device %d", dev);
        g_scratch_ptr[dev] = ptr;
    }
    *out = g_scratch_ptr[dev];
    return MF_OK;
}

}  // namespace mf

using namespace mf;

extern "C" {

size_t mf_sort_by_count_workspace_bytes(uint32_t n)
{
    if (n == 0) return 0;
    size_t tmp = 0, total = 0;
    return sort_layout(n, &tmp, &total) == MF_OK ? total : 0;
}
int mf_sort_by_count_ws(uint32_t* cnt, uint32_t* idx, uint32_t n, void* workspace, size_t workspace_bytes, void* stream)
{
    if (n == 0) return MF_OK;
    if (!cnt || !idx || !workspace) return invalid("mf_sort_by_count_ws: null pointer");
    if (reinterpret_cast<uintptr_t>(workspace) % kAlign) return invalid("mf_sort_by_count_ws: the workspace must be 256-byte aligned");
    size_t tmp = 0, total = 0;
    if (int rc = sort_layout(n, &tmp, &total)) return rc;
    if (workspace_bytes < total) return invalid("mf_sort_by_count_ws: the workspace holds %zu bytes, %u counts need %zu (mf_sort_by_count_workspace_bytes)", workspace_bytes, n, total);
    return sort_in(cnt, idx, n, static_cast<uint8_t*>(workspace), tmp, as_stream(stream));
}
int mf_sort_by_count(uint32_t* cnt, uint32_t* idx, uint32_t n, void* stream)
{
    if (n == 0) return MF_OK;
    if (!cnt || !idx) return invalid("mf_sort_by_count: null pointer");
    size_t tmp = 0, total = 0;
    if (int rc = sort_layout(n, &tmp, &total)) return rc;
    DeviceBuffers b;
    if (int rc = check_hip(hipMalloc(&b.ptr[0], total), "mf_sort_by_count: hipMalloc")) return rc;
    if (int rc = sort_in(cnt, idx, n, static_cast<uint8_t*>(b.ptr[0]), tmp, as_stream(stream))) return rc;
    return check_hip(hipStreamSynchronize(as_stream(stream)), "mf_sort_by_count: synchronize");      // the workspace is freed on return
}
uint32_t mf_sort_by_count_static_max(void) { return kStaticSortMax; }
int mf_sort_by_count_static(uint32_t* cnt, uint32_t* idx, uint32_t n, void* stream)
{
    if (n == 0) return MF_OK;
    if (!cnt || !idx) return invalid("mf_sort_by_count_static: null pointer");
    if (n > kStaticSortMax) return invalid("mf_sort_by_count_static: %u counts, the library's own scratch holds at most %u (use mf_sort_by_count_ws with a workspace)", n, kStaticSortMax);
    size_t tmp = 0, total = 0;
    if (int rc = sort_layout(n, &tmp, &total)) return rc;
    if (total > kStaticScratchBytes) return invalid("mf_sort_by_count_static: %u counts need %zu bytes of scratch, the library's own holds %zu", n, total, kStaticScratchBytes);
    void* ptr = nullptr;
    if (int rc = static_scratch(&ptr)) return rc;
    // nothing in the scratch has to start at zero: the sort writes its output buffers before it reads them and rocPRIM
    // initialises what it keeps in its temporary storage
    return sort_in(cnt, idx, n, static_cast<uint8_t*>(ptr), tmp, as_stream(stream));
}

size_t mf_shuffle_ratings_workspace_bytes(uint32_t n) { return n == 0 ? 0 : shuffle_plan(n).total; }
int mf_shuffle_ratings_ws(const mf_node* in, mf_node* out, uint32_t n, uint64_t seed, void* workspace, size_t workspace_bytes, void* stream)
{
    if (n == 0) return MF_OK;
    if (!in || !out || in == out) return invalid("mf_shuffle_ratings: null or aliased buffers");
    if (!workspace || reinterpret_cast<uintptr_t>(workspace) % kAlign) return invalid("mf_shuffle_ratings_ws: the workspace must be non-null and 256-byte aligned");
    const ShufflePlan p = shuffle_plan(n);
    if (workspace_bytes < p.total) return invalid("mf_shuffle_ratings_ws: the workspace holds %zu bytes, %u ratings need %zu (mf_shuffle_ratings_workspace_bytes)", workspace_bytes, n, p.total);
    hipStream_t s = as_stream(stream);
    uint8_t* ws = static_cast<uint8_t*>(workspace);
    PassArgs a = {};
    a.nodes = reinterpret_cast<const Node3*>(in); a.n = n; a.base = mix64(seed ^ 0x53485546464C4521ull); a.segs = 1;
    for (int l = 0; l < 2; ++l) {
        a.bits = l ? p.bits2 : p.bits1;
        if (!a.bits) break;
        a.chunks = l ? p.chunks2 : p.chunks1;
        a.moved_out = reinterpret_cast<uint4*>(ws + p.moved[l]);
        a.table = reinterpret_cast<uint32_t*>(ws + p.table[l]); a.bucket_start = reinterpret_cast<uint32_t*>(ws + p.start[l]);
        auto pass = [&](auto Block, auto count, auto partition) -> int {
            const dim3 grid(a.segs * a.chunks), block(decltype(Block)::value);
            if (int rc = check_hip(hipFuncSetAttribute(reinterpret_cast<const void*>(partition), hipFuncAttributeMaxDynamicSharedMemorySize, (int)partition_lds(a.bits)),
                                   "hipFuncSetAttribute(MaxDynamicSharedMemorySize)")) return rc;
            hipLaunchKernelGGL(count, grid, block, (size_t)4 << a.bits, s, a);
            hipLaunchKernelGGL(shuffle_place_kernel, dim3(a.segs), dim3(kShufBlock), place_lds(a.bits), s, a);
            hipLaunchKernelGGL(partition, grid, block, partition_lds(a.bits), s, a);
            return MF_OK;
        };
        auto either = [&](auto Moved) {
            constexpr bool moved = decltype(Moved)::value;
            return a.bits <= kLargeTileBits ? pass(std::integral_constant<int, 1024>(), shuffle_count_kernel<1024>, shuffle_partition_kernel<1024, moved>)
                                            : pass(std::integral_constant<int, 512>(), shuffle_count_kernel<512>, shuffle_partition_kernel<512, moved>);
        };
        if (int rc = l ? either(std::true_type()) : either(std::false_type())) return rc;
        if (int rc = launch_status("mf_shuffle_ratings: partition")) return rc;
        a.moved = a.moved_out; a.seg_start = a.bucket_start;
        a.segs <<= a.bits; a.skip += a.bits;
    }
    hipLaunchKernelGGL((a.moved ? shuffle_finish_kernel<true> : shuffle_finish_kernel<false>), dim3(a.segs), dim3(kShufBlock), 0, s, a.moved, a.nodes, reinterpret_cast<Node3*>(out), n, a.base, a.skip, a.seg_start, a.segs);
    return launch_status("mf_shuffle_ratings: order");
}
int mf_shuffle_ratings(const mf_node* in, mf_node* out, uint32_t n, uint64_t seed, void* stream)
{
    if (n == 0) return MF_OK;
    if (!in || !out || in == out) return invalid("mf_shuffle_ratings: null or aliased buffers");
    const size_t total = shuffle_plan(n).total;
    DeviceBuffers b;
    if (int rc = check_hip(hipMalloc(&b.ptr[0], total), "mf_shuffle_ratings: hipMalloc")) return rc;
    if (int rc = mf_shuffle_ratings_ws(in, out, n, seed, b.ptr[0], total, stream)) return rc;
    return check_hip(hipStreamSynchronize(as_stream(stream)), "mf_shuffle_ratings: synchronize");      // the workspace is freed on return
}

}  // extern "C"
