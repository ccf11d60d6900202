// LBVH build on gfx950: primitive centres/boxes, scene box, 63-bit Morton
// codes, LDS-staged stable LSD radix sort, Karras hierarchy and node boxes.  Reference: Tracer/AcceleratorLBVH.{hpp,cu}, Tracer/AcceleratorWork.kt.h.
#include "common.h"
#include "lbvh.h"

#include <algorithm>
#include <mutex>
#include <string>

namespace mray
{

// ---------------------------------------------------------------------------
// KCGenPrimCenters + KCGeneratePrimAABBs (AcceleratorWork.kt.h:5-123):
// one thread per triangle.  Centre = p0*k + p1*k + p2*k, k = 0.333333333
// (PrimitiveDefaultTriangle.hpp:107-115), box = component min/max.
// ---------------------------------------------------------------------------
__global__ void __launch_bounds__(kTPB)
KCPrimCentersAabbs(const float* __restrict__ pos, const uint32_t* __restrict__ idx,
                   uint32_t n, float* __restrict__ centers, float* __restrict__ aabbs)
{
    uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
    if(t >= n) return;
    uint32_t i0 = idx[3 * t + 0], i1 = idx[3 * t + 1], i2 = idx[3 * t + 2];
    V3 p0 = {pos[3 * i0], pos[3 * i0 + 1], pos[3 * i0 + 2]};
    V3 p1 = {pos[3 * i1], pos[3 * i1 + 1], pos[3 * i1 + 2]};
    V3 p2 = {pos[3 * i2], pos[3 * i2 + 1], pos[3 * i2 + 2]};
    const float k = 0.333333333f;
    V3 c = (p0 * k + p1 * k) + p2 * k;
    if(centers)
    {
        centers[3 * t + 0] = c.x;
        centers[3 * t + 1] = c.y;
        centers[3 * t + 2] = c.z;
    }
    if(aabbs)
    {
        float* b = aabbs + 6 * size_t(t);
        b[0] = MinF(MinF(p0.x, p1.x), p2.x);
        b[1] = MinF(MinF(p0.y, p1.y), p2.y);
        b[2] = MinF(MinF(p0.z, p1.z), p2.z);
        b[3] = MaxF(MaxF(p0.x, p1.x), p2.x);
        b[4] = MaxF(MaxF(p0.y, p1.y), p2.y);
        b[5] = MaxF(MaxF(p0.z, p1.z), p2.z);
    }
}

// ---------------------------------------------------------------------------
// Scene box: two-level min/max reduction (exact, order-free).
// ---------------------------------------------------------------------------
static constexpr uint32_t kReduceBlocks = 1024;

__global__ void __launch_bounds__(kTPB)
KCReduceAabbPartial(const float* __restrict__ aabbs, uint32_t n, float* __restrict__ partial)
{
    __shared__ float s[6][kTPB];
    float b[6] = {INFINITY, INFINITY, INFINITY, -INFINITY, -INFINITY, -INFINITY};
    for(uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x)
    {
        const float* a = aabbs + 6 * size_t(i);
        for(int k = 0; k < 3; k++)
        {
            b[k] = MinF(b[k], a[k]);
            b[3 + k] = MaxF(b[3 + k], a[3 + k]);
        }
    }
    for(int k = 0; k < 6; k++) s[k][threadIdx.x] = b[k];
    __syncthreads();
    for(uint32_t st = blockDim.x / 2; st > 0; st >>= 1)
    {
        if(threadIdx.x < st)
        {
            for(int k = 0; k < 3; k++)
            {
                s[k][threadIdx.x] = MinF(s[k][threadIdx.x], s[k][threadIdx.x + st]);
                s[3 + k][threadIdx.x] = MaxF(s[3 + k][threadIdx.x], s[3 + k][threadIdx.x + st]);
            }
        }
        __syncthreads();
    }
    if(threadIdx.x < 6) partial[6 * blockIdx.x + threadIdx.x] = s[threadIdx.x][0];
}

// ---------------------------------------------------------------------------
// KCGenMortonCode (AcceleratorLBVH.cu:96-168), bit-exact: float offset from
// the box minimum clamped at 0, double product with 2^21 / maxSide, rounded
// back to float, lroundf, clamp to [0, 2^21 - 1], Compose3D<uint64_t>.
// ---------------------------------------------------------------------------
__device__ __forceinline__ uint64_t Expand3D64(uint32_t v)
{
    uint64_t x = v;
    x &= 0x1fffff;
    x = (x | x << 32) & 0x001f00000000ffffull;
    x = (x | x << 16) & 0x001f0000ff0000ffull;
    x = (x | x << 8) & 0x100f00f00f00f00full;
    x = (x | x << 4) & 0x10c30c30c30c30c3ull;
    x = (x | x << 2) & 0x1249249249249249ull;
    return x;
}
__device__ __forceinline__ uint32_t Expand3D32(uint32_t x)
{
    x &= 0x000003ff;
    x = (x ^ (x << 16)) & 0xff0000ff;
    x = (x ^ (x << 8)) & 0x0300f00f;
    x = (x ^ (x << 4)) & 0x030c30c3;
    x = (x ^ (x << 2)) & 0x09249249;
    return x;
}

template<uint32_t BITS>
__device__ __forceinline__ void Quantize(const float* __restrict__ c, const float* __restrict__ box,
                                         uint32_t q[3])
{
    float sx = box[3] - box[0], sy = box[4] - box[1], sz = box[5] - box[2];
    float maxSide = sx;
    if(sy > maxSide) maxSide = sy;
    if(sz > maxSide) maxSide = sz;
    const double sliceCount = double(1ull << BITS);
    double deltaRecip = sliceCount / double(maxSide);
    const uint32_t last = (1u << BITS) - 1u;
    for(int k = 0; k < 3; k++)
    {
        float d = MaxF(c[k] - box[k], 0.0f);
        float qf = float(double(d) * deltaRecip);
        uint32_t qi = uint32_t(int32_t(lroundf(qf)));
        q[k] = (qi > last) ? last : qi;
    }
}

__global__ void __launch_bounds__(kTPB)
KCMorton63(const float* __restrict__ centers, uint32_t n, const float* __restrict__ box,
           uint64_t* __restrict__ codes)
{
    uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if(i >= n) return;
    float c[3] = {centers[3 * i], centers[3 * i + 1], centers[3 * i + 2]};
    float b[6];
    for(int k = 0; k < 6; k++) b[k] = box[k];
    uint32_t q[3];
    Quantize<21>(c, b, q);
    codes[i] = Expand3D64(q[0]) | (Expand3D64(q[1]) << 1) | (Expand3D64(q[2]) << 2);
}

__global__ void __launch_bounds__(kTPB)
KCMorton30(const float* __restrict__ centers, uint32_t n, const float* __restrict__ box,
           uint32_t* __restrict__ codes)
{
    uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if(i >= n) return;
    float c[3] = {centers[3 * i], centers[3 * i + 1], centers[3 * i + 2]};
    float b[6];
    for(int k = 0; k < 6; k++) b[k] = box[k];
    uint32_t q[3];
    Quantize<10>(c, b, q);
    codes[i] = Expand3D32(q[0]) | (Expand3D32(q[1]) << 1) | (Expand3D32(q[2]) << 2);
}

// ---------------------------------------------------------------------------
// Stable LSD radix sort of (u64 key, u32 value), 8 bits per pass, in one of
// two forms by count:
//
// Up to 12288 pairs: one workgroup of 16 waves keeps every pair in registers
// and permutes them through LDS between passes (KCRadixSortOneGroup), one
// launch and no global traffic between passes.  Bound by the latency of its
// serial ranking rounds.  9,800 pairs: 24 launches, 195 us -> one launch,
// 69 us.  Beyond that the 160 KiB of LDS are full.
//
// More: per pass a tile histogram, a scan and a scatter.
//   KCRadixHist     counts of each tile, digit-major
//   KCRadixScan     one workgroup per digit scans its row over the tiles (the
//                   256 digit totals are scanned by every scatter block)
//   KCRadixScatter  ranks a tile, sorts it by digit in LDS and writes it out,
//                   so that a digit's keys leave in one run: bound by HBM
//                   (24 B per pair and pass)
// The scan was one workgroup walking all 256 x tiles counts: 247 us a pass
// at 2.25 M pairs, now 4.8 us; the scatter 40.1 -> 16.0 us.
//
// Ranking (both forms): a wave owns 64 R consecutive pairs and takes them 64
// at a time; 8 ballots give each lane the lanes with its digit (its peers),
// and a per-wave count table in LDS gives the pairs of that digit in the
// wave's earlier rounds, so equal digits keep input order.
// ---------------------------------------------------------------------------
static constexpr uint32_t kRsThreads = 256;
static constexpr uint32_t kRsWaves = kRsThreads / 64;
static constexpr uint32_t kRsOneThreads = 1024;
static constexpr uint32_t kRsOneMax = kRsOneThreads * 12u;
// Rounds per wave of a tile (256 pairs each).  A tile's rounds are serial and
// its pairs fill LDS (8 workgroups of 4 rounds share a CU, 4 of 8, 3 of 12,
// 2 of 16), so tiles grow only as the count fills the 256 CUs; larger tiles
// have longer digit runs and fewer histogram rows.  Whole sorts with 8 / 12 /
// 16 rounds: 2^19 pairs 123 / 142 / 163 us, 10^6 149 / 163 / 167, 2.25 M 229 /
// 212 / 270, 8 M 688 / 614 / 611; 4 rounds below 2^19: 300 K 111 us.
static constexpr uint32_t kRsMidFrom = 1u << 19, kRsLargeFrom = 1u << 21;
static constexpr uint32_t RsRounds(uint32_t n) { return (n < kRsMidFrom) ? 4u : (n < kRsLargeFrom) ? 8u : 12u; }
static constexpr uint32_t RsTile(uint32_t n) { return kRsThreads * RsRounds(n); }

// Lanes of the wave whose key has this lane's digit (valid lanes only).
__device__ __forceinline__ uint64_t DigitPeers(uint32_t digit, bool valid)
{
    const uint64_t in = __ballot(valid);
    uint32_t lo = uint32_t(in), hi = uint32_t(in >> 32);
    #pragma unroll
    for(uint32_t b = 0; b < 8; b++)
    {
        const uint32_t one = (digit >> b) & 1u;
        const uint64_t bb = __ballot(one != 0u);
        const uint32_t mask = 0u - one;
        lo &= ~(uint32_t(bb) ^ mask);
        hi &= ~(uint32_t(bb >> 32) ^ mask);
    }
    return (uint64_t(hi) << 32) | lo;
}

// One ranking round: pairs of this digit that the wave met before this lane's
// (in earlier rounds and in lower lanes); `cnt` is the wave's count table.
template<class C>
__device__ __forceinline__ uint32_t RankRound(C* cnt, uint32_t digit, bool valid, uint64_t ltMask)
{
    const uint64_t peers = DigitPeers(digit, valid);
    const uint32_t rank = uint32_t(__popcll(peers & ltMask));
    const uint32_t before = cnt[digit];
    __builtin_amdgcn_wave_barrier();
    if(valid && rank == 0) cnt[digit] = C(before + uint32_t(__popcll(peers)));
    __builtin_amdgcn_wave_barrier();
    return before + rank;
}

// Exclusive scan over the 256 threads of waves 0..3 (every thread of the
// block calls it; threads past 255 only join the barriers).
__device__ __forceinline__ uint32_t ScanDigits(uint32_t v, uint32_t* waveSum)
{
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    uint32_t incl = v;
    for(uint32_t o = 1; o < 64; o <<= 1)
    {
        const uint32_t up = __shfl_up(incl, o);
        if(lane >= o) incl += up;
    }
    if(wave < 4 && lane == 63) waveSum[wave] = incl;
    __syncthreads();
    uint32_t excl = incl - v;
    for(uint32_t w = 0; w < 3; w++)
        if(w < wave) excl += waveSum[w];
    __syncthreads();
    return excl;
}

template<uint32_t R>
__global__ void __launch_bounds__(kRsThreads)
KCRadixHist(const uint64_t* __restrict__ keys, uint32_t n, uint32_t shift, uint32_t numTiles,
            uint32_t* __restrict__ hist)
{
    __shared__ uint32_t h[256];
    h[threadIdx.x] = 0;
    __syncthreads();
    const uint32_t base = blockIdx.x * kRsThreads * R;
    #pragma unroll
    for(uint32_t r = 0; r < R; r++)
    {
        const uint32_t i = base + r * kRsThreads + threadIdx.x;
        if(i < n) atomicAdd(&h[uint32_t(keys[i] >> shift) & 255u], 1u);
    }
    __syncthreads();
    hist[size_t(threadIdx.x) * numTiles + blockIdx.x] = h[threadIdx.x];
}

// Block d: exclusive scan of digit d's counts over the tiles, in place, and
// the digit's total.
__global__ void __launch_bounds__(kRsThreads)
KCRadixScan(uint32_t* __restrict__ hist, uint32_t numTiles, uint32_t* __restrict__ total)
{
    __shared__ uint32_t waveSum[4];
    __shared__ uint32_t blockSum;
    uint32_t* row = hist + size_t(blockIdx.x) * numTiles;
    uint32_t carry = 0;
    for(uint32_t base = 0; base < numTiles; base += kRsThreads)
    {
        const uint32_t i = base + threadIdx.x;
        const uint32_t v = (i < numTiles) ? row[i] : 0u;
        const uint32_t excl = ScanDigits(v, waveSum);
        if(i < numTiles) row[i] = carry + excl;
        if(threadIdx.x == kRsThreads - 1u) blockSum = excl + v;
        __syncthreads();
        carry += blockSum;
        __syncthreads();
    }
    if(threadIdx.x == 0) total[blockIdx.x] = carry;
}

template<uint32_t R>
__global__ void __launch_bounds__(kRsThreads)
KCRadixScatter(const uint64_t* __restrict__ keysIn, const uint32_t* __restrict__ valsIn,
               uint64_t* __restrict__ keysOut, uint32_t* __restrict__ valsOut, uint32_t n,
               uint32_t shift, uint32_t numTiles, const uint32_t* __restrict__ histScan,
               const uint32_t* __restrict__ total)
{
    constexpr uint32_t kTile = kRsThreads * R;
    __shared__ uint64_t sKey[kTile];
    __shared__ uint32_t sVal[kTile];
    __shared__ uint32_t cnt[kRsWaves][256];
    __shared__ uint32_t start[256];     // first local position of a digit
    __shared__ uint32_t outBase[256];   // its first output position - start
    __shared__ uint32_t waveSum[4];
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
    const uint64_t ltMask = (lane == 0) ? 0ull : ((~0ull) >> (64 - lane));
    const uint32_t tileStart = blockIdx.x * kTile;
    const uint32_t tileCount = min(kTile, n - tileStart);
    const uint32_t first = wave * 64u * R + lane;
    uint64_t key[R];
    uint32_t val[R], rank[R];
    #pragma unroll
    for(uint32_t r = 0; r < R; r++)
    {
        const uint32_t k = first + r * 64u;
        key[r] = (k < tileCount) ? keysIn[tileStart + k] : 0ull;
        val[r] = (k < tileCount) ? valsIn[tileStart + k] : 0u;
    }
    const uint32_t tileOff = histScan[size_t(tid) * numTiles + blockIdx.x];
    const uint32_t digitOff = ScanDigits(total[tid], waveSum);
    for(uint32_t w = 0; w < kRsWaves; w++) cnt[w][tid] = 0;
    __syncthreads();
    #pragma unroll
    for(uint32_t r = 0; r < R; r++)
        rank[r] = RankRound(cnt[wave], uint32_t(key[r] >> shift) & 255u, first + r * 64u < tileCount, ltMask);
    __syncthreads();
    uint32_t acc = 0;
    for(uint32_t w = 0; w < kRsWaves; w++)
    {
        const uint32_t c = cnt[w][tid];
        cnt[w][tid] = acc;
        acc += c;
    }
    const uint32_t s = ScanDigits(acc, waveSum);
    start[tid] = s;
    outBase[tid] = digitOff + tileOff - s;
    __syncthreads();
    #pragma unroll
    for(uint32_t r = 0; r < R; r++)
    {
        if(first + r * 64u >= tileCount) continue;
        const uint32_t d = uint32_t(key[r] >> shift) & 255u;
        const uint32_t at = start[d] + cnt[wave][d] + rank[r];
        sKey[at] = key[r];
        sVal[at] = val[r];
    }
    __syncthreads();
    #pragma unroll
    for(uint32_t r = 0; r < R; r++)
    {
        const uint32_t j = r * kRsThreads + tid;
        if(j >= tileCount) continue;
        const uint64_t k = sKey[j];
        const uint32_t dst = outBase[uint32_t(k >> shift) & 255u] + j;
        keysOut[dst] = k;
        valsOut[dst] = sVal[j];
    }
}

// The whole sort of at most 1024 R pairs in one workgroup, in place.
template<uint32_t R>
__global__ void __launch_bounds__(kRsOneThreads)
KCRadixSortOneGroup(uint64_t* __restrict__ keys, uint32_t* __restrict__ vals, uint32_t n)
{
    constexpr uint32_t kWaves = kRsOneThreads / 64u;
    __shared__ uint64_t sKey[kRsOneThreads * R];
    __shared__ uint32_t sVal[kRsOneThreads * R];
    __shared__ uint16_t cnt[kWaves][256];     // counts and positions stay below 12288
    __shared__ uint16_t start[256];
    __shared__ uint32_t waveSum[4];
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
    const uint64_t ltMask = (lane == 0) ? 0ull : ((~0ull) >> (64 - lane));
    // the pairs in use split evenly over the waves, in 64s
    const uint32_t rounds = (n + kRsOneThreads - 1u) / kRsOneThreads;
    const uint32_t first = wave * 64u * rounds + lane;
    uint64_t key[R];
    uint32_t val[R], rank[R];
    #pragma unroll
    for(uint32_t r = 0; r < R; r++)
    {
        const uint32_t k = first + r * 64u;
        const bool in = r < rounds && k < n;
        key[r] = in ? keys[k] : 0ull;
        val[r] = in ? vals[k] : 0u;
    }
    for(uint32_t shift = 0; shift < 64u; shift += 8u)
    {
        for(uint32_t e = tid; e < kWaves * 256u; e += kRsOneThreads) cnt[0][e] = 0;
        __syncthreads();
        #pragma unroll
        for(uint32_t r = 0; r < R; r++)
            if(r < rounds)
                rank[r] = RankRound(cnt[wave], uint32_t(key[r] >> shift) & 255u, first + r * 64u < n, ltMask);
        __syncthreads();
        uint32_t acc = 0;
        if(tid < 256u)
            for(uint32_t w = 0; w < kWaves; w++)
            {
                const uint32_t c = cnt[w][tid];
                cnt[w][tid] = uint16_t(acc);
                acc += c;
            }
        const uint32_t s = ScanDigits(acc, waveSum);
        if(tid < 256u) start[tid] = uint16_t(s);
        __syncthreads();
        #pragma unroll
        for(uint32_t r = 0; r < R; r++)
        {
            if(r >= rounds || first + r * 64u >= n) continue;
            const uint32_t d = uint32_t(key[r] >> shift) & 255u;
            const uint32_t at = uint32_t(start[d]) + cnt[wave][d] + rank[r];
            sKey[at] = key[r];
            sVal[at] = val[r];
        }
        __syncthreads();
        #pragma unroll
        for(uint32_t r = 0; r < R; r++)
        {
            const uint32_t k = first + r * 64u;
            if(r >= rounds || k >= n) continue;
            key[r] = sKey[k];
            val[r] = sVal[k];
        }
    }
    #pragma unroll
    for(uint32_t r = 0; r < R; r++)
    {
        const uint32_t k = first + r * 64u;
        if(r >= rounds || k >= n) continue;
        keys[k] = key[r];
        vals[k] = val[r];
    }
}

// ---------------------------------------------------------------------------
// KCConstructLBVHInternalNodes (AcceleratorLBVH.cu:170-299), Karras 2012
// Fig. 4 with the reference's Delta (equal codes fall back to the index XOR,
// AcceleratorLBVH.cu:69-94).  Also records each node's leaf range.
// ---------------------------------------------------------------------------
// strict = 0: the reference's fallback, clz(i ^ j) on equal codes.  It can
// rank a run of equal codes below neighbours that differ only in low bits,
// which breaks the Karras prefix order (some nodes/leaves get no parent).
// strict = 1: the key is (code, index), so equal codes rank above every
// distinct pair (64 + clz32(i ^ j)); used to rebuild such inputs.
//
// Bound by the latency of the search's dependent code reads; most nodes span
// a few leaves, so a block keeps the codes around its own in LDS and only
// the searches of large nodes leave it.
static constexpr int32_t kCodeHalo = 128;
static constexpr int32_t kCodeWindow = int32_t(kTPB) + 2 * kCodeHalo;
__device__ __forceinline__ int32_t Delta(const uint64_t* __restrict__ codes, const uint64_t* window,
                                         int32_t windowFirst, int32_t n, int32_t i, uint64_t l,
                                         int32_t j, uint32_t strict)
{
    if(j < 0 || j >= n) return -1;
    const uint32_t at = uint32_t(j - windowFirst);
    uint64_t r = (at < uint32_t(kCodeWindow)) ? window[at] : codes[j];
    if(l == r)
    {
        if(strict) return 64 + int32_t(__clz(uint32_t(i ^ j)));
        l = uint64_t(i);
        r = uint64_t(j);
    }
    uint64_t d = l ^ r;
    return (d == 0) ? 64 : int32_t(__clzll(d));
}

// ---------------------------------------------------------------------------
// Node boxes (KCUnionLBVHBoundingBoxes, AcceleratorLBVH.cu:301-435).  A node's
// box is the union of the leaf boxes of its leaf-order range, and min / max
// do not depend on the order, so no node has to wait for its children: the
// leaf boxes are gathered in leaf order and reduced to levels of 4, 16, 64,
// ... consecutive leaves, and each node unites the few level entries that
// tile its range, in the kernel that found the range.  The bottom-up climb
// this replaces paid an agent-scope fence (an L2 write-back across the XCDs)
// per step: 11.1 ms at 2.25 M leaves, now 43 us for the levels and
// 116 us for ranges and boxes.  Four leaves per entry: a range takes at
// most 3 entries per level and end, and a wave waits for its longest node.
// ---------------------------------------------------------------------------
struct alignas(16) LevelBox
{
    float4 lo, hi;       // xyz, w unused
};
static constexpr uint32_t kBoxLevels = 17;       // 4^16 = 2^32 leaves
static constexpr uint32_t kLevelsPerBlock = 5;   // levels 1..5: 1024 leaves
static constexpr uint32_t kLevelTPB = 1024;
struct BoxLevels
{
    LevelBox* base;
    size_t off[kBoxLevels];
    uint32_t count[kBoxLevels];
    uint32_t levels;     // the last one holds a single entry
};

// Entries of every level of n leaves (off / count may be null).
static size_t BoxLevelEntries(uint32_t n, BoxLevels* out)
{
    size_t total = 0;
    uint32_t l = 0;
    for(uint32_t c = n;; c = DivUp(c, 4u), l++)
    {
        if(out) { out->off[l] = total; out->count[l] = c; out->levels = l + 1; }
        total += c;
        if(c <= 1) break;
    }
    return total;
}

struct Box6
{
    float lo[3], hi[3];
};
__device__ __forceinline__ Box6 EmptyBox()
{
    return {{INFINITY, INFINITY, INFINITY}, {-INFINITY, -INFINITY, -INFINITY}};
}
__device__ __forceinline__ void Unite(Box6& b, const LevelBox& e)
{
    b.lo[0] = MinF(b.lo[0], e.lo.x); b.lo[1] = MinF(b.lo[1], e.lo.y); b.lo[2] = MinF(b.lo[2], e.lo.z);
    b.hi[0] = MaxF(b.hi[0], e.hi.x); b.hi[1] = MaxF(b.hi[1], e.hi.y); b.hi[2] = MaxF(b.hi[2], e.hi.z);
}
__device__ __forceinline__ LevelBox ToLevel(const Box6& b)
{
    return {make_float4(b.lo[0], b.lo[1], b.lo[2], 0.0f), make_float4(b.hi[0], b.hi[1], b.hi[2], 0.0f)};
}
__device__ __forceinline__ void UniteLanes(Box6& b, int mask)
{
    #pragma unroll
    for(int k = 0; k < 3; k++)
    {
        b.lo[k] = MinF(b.lo[k], __shfl_xor(b.lo[k], mask));
        b.hi[k] = MaxF(b.hi[k], __shfl_xor(b.hi[k], mask));
    }
}

// Levels 0..5 of 1024 leaves per block; also marks every node's parent unset.
__global__ void __launch_bounds__(kLevelTPB)
KCLeafLevels(const uint32_t* __restrict__ leafOrder, const float* __restrict__ leafAabbs, uint32_t n,
             BoxLevels lv, uint32_t* __restrict__ nodes)
{
    static_assert(kLevelTPB == 1024 && kLevelsPerBlock == 5, "five levels of 4 per block");
    __shared__ LevelBox waveBox[kLevelTPB / 64];
    const uint32_t p = blockIdx.x * blockDim.x + threadIdx.x;
    Box6 b = EmptyBox();
    if(p < n)
    {
        const float* src = leafAabbs + 6 * size_t(leafOrder[p]);
        #pragma unroll
        for(int k = 0; k < 3; k++) { b.lo[k] = src[k]; b.hi[k] = src[3 + k]; }
        lv.base[p] = ToLevel(b);
        if(n == 1 || p < n - 1u) nodes[size_t(p) * 3 + 2] = kInvalid;
    }
    #pragma unroll
    for(uint32_t l = 1; l <= 3; l++)
    {
        UniteLanes(b, 1 << (2 * l - 2));
        UniteLanes(b, 1 << (2 * l - 1));
        if(l < lv.levels && p < n && (p & ((1u << (2 * l)) - 1u)) == 0u)
            lv.base[lv.off[l] + (p >> (2 * l))] = ToLevel(b);
    }
    if(lv.levels <= 4u) return;
    if((threadIdx.x & 63u) == 0u) waveBox[threadIdx.x >> 6] = ToLevel(b);
    __syncthreads();
    if(threadIdx.x >= 64u) return;
    // the block's 16 waves are 16 consecutive entries of level 3
    b = EmptyBox();
    if(threadIdx.x < kLevelTPB / 64u) Unite(b, waveBox[threadIdx.x]);
    UniteLanes(b, 1);
    UniteLanes(b, 2);
    const uint32_t q = blockIdx.x * 4u + (threadIdx.x >> 2);
    if(threadIdx.x < kLevelTPB / 64u && (threadIdx.x & 3u) == 0u && q < lv.count[4])
        lv.base[lv.off[4] + q] = ToLevel(b);
    UniteLanes(b, 4);
    UniteLanes(b, 8);
    if(threadIdx.x == 0 && lv.levels > 5u) lv.base[lv.off[5] + blockIdx.x] = ToLevel(b);
}

// Levels 6 and up, by one workgroup, three levels between barriers: a wave
// reads 64 consecutive entries and unites them in groups of 4, 16 and 64.
__global__ void __launch_bounds__(1024)
KCTopLevels(BoxLevels lv)
{
    for(uint32_t l = kLevelsPerBlock; l + 1u < lv.levels; l += 3u)
    {
        const LevelBox* src = lv.base + lv.off[l];
        const uint32_t count = lv.count[l];
        for(uint32_t p = threadIdx.x; p < ((count + 63u) & ~63u); p += blockDim.x)
        {
            Box6 b = EmptyBox();
            if(p < count) Unite(b, src[p]);
            #pragma unroll
            for(uint32_t k = 1; k <= 3; k++)
            {
                UniteLanes(b, 1 << (2 * k - 2));
                UniteLanes(b, 1 << (2 * k - 1));
                if(l + k < lv.levels && p < count && (p & ((1u << (2 * k)) - 1u)) == 0u)
                    lv.base[lv.off[l + k] + (p >> (2 * k))] = ToLevel(b);
            }
        }
        __syncthreads();
    }
}

// Union of leaves [first, last] of the leaf order.
__device__ __forceinline__ Box6 RangeBox(const BoxLevels& lv, uint32_t first, uint32_t last)
{
    Box6 b = EmptyBox();
    uint32_t a = first, e = last + 1u;
    for(uint32_t l = 0; a < e; l++)
    {
        const LevelBox* at = lv.base + lv.off[l];
        // up to three entries at each end, their loads in flight together:
        // past the end's last entry, that one is read again
        const uint32_t na = min((4u - (a & 3u)) & 3u, e - a);
        if(na)
        {
            const LevelBox x = at[a], y = at[a + min(1u, na - 1u)], z = at[a + na - 1u];
            Unite(b, x); Unite(b, y); Unite(b, z);
            a += na;
        }
        const uint32_t ne = min(e & 3u, e - a);
        if(ne)
        {
            const LevelBox x = at[e - 1u], y = at[e - min(2u, ne)], z = at[e - ne];
            Unite(b, x); Unite(b, y); Unite(b, z);
            e -= ne;
        }
        a >>= 2;
        e >>= 2;
    }
    return b;
}

__device__ __forceinline__ int32_t DivUpI(int32_t v, int32_t d) { return (v + d - 1) / d; }

__device__ __forceinline__ void StoreBox(float* __restrict__ dst, const Box6& b)
{
    #pragma unroll
    for(int k = 0; k < 3; k++) { dst[k] = b.lo[k]; dst[3 + k] = b.hi[k]; }
}

__global__ void __launch_bounds__(kTPB)
KCKarras(const uint64_t* __restrict__ codes, const uint32_t* __restrict__ leafOrder, int32_t n,
         uint32_t* __restrict__ nodes, uint32_t* __restrict__ nodeRange, BoxLevels lv,
         float* __restrict__ boxes, uint32_t strict)
{
    int32_t i = int32_t(blockIdx.x * blockDim.x + threadIdx.x);
    if(n == 1)
    {
        if(i == 0)
        {
            nodes[0] = kLeafFlag | 0u;
            nodes[1] = kInvalid;
            nodes[2] = kInvalid;
            if(nodeRange) { nodeRange[0] = 0; nodeRange[1] = 0; }
            StoreBox(boxes, RangeBox(lv, 0u, 0u));
        }
        return;
    }
    __shared__ uint64_t window[kCodeWindow];
    const int32_t w0 = int32_t(blockIdx.x * blockDim.x) - kCodeHalo;
    for(int32_t e = int32_t(threadIdx.x); e < kCodeWindow; e += int32_t(kTPB))
        window[e] = codes[max(0, min(n - 1, w0 + e))];
    __syncthreads();
    if(i >= n - 1) return;
    const uint64_t code = window[i - w0];
    auto delta = [&](int32_t j) { return Delta(codes, window, w0, n, i, code, j, strict); };
    int32_t diff = delta(i + 1) - delta(i - 1);
    int32_t d = (diff < 0) ? -1 : 1;
    int32_t deltaMin = delta(i - d);
    int32_t lMax = 2;
    while(delta(i + lMax * d) > deltaMin) lMax <<= 1;
    int32_t l = 0;
    for(int32_t t = lMax >> 1; t != 0; t >>= 1)
        if(delta(i + (l + t) * d) > deltaMin) l += t;
    int32_t j = i + l * d;
    int32_t s = 0;
    int32_t deltaNode = delta(j);
    for(int32_t t = DivUpI(l, 2); t != 0; t = (t == 1) ? 0 : DivUpI(t, 2))
        if(delta(i + (s + t) * d) > deltaNode) s += t;
    int32_t gamma = i + s * d + min(d, 0);

    uint32_t* me = nodes + size_t(i) * 3;
    int32_t lo = min(i, j), hi = max(i, j);
    if(lo == gamma)
    {
        me[0] = kLeafFlag | leafOrder[gamma];
    }
    else
    {
        me[0] = uint32_t(gamma);
        nodes[size_t(gamma) * 3 + 2] = uint32_t(i);
    }
    if(hi == gamma + 1)
    {
        me[1] = kLeafFlag | leafOrder[gamma + 1];
    }
    else
    {
        me[1] = uint32_t(gamma + 1);
        nodes[size_t(gamma + 1) * 3 + 2] = uint32_t(i);
    }
    if(nodeRange)
    {
        nodeRange[2 * i + 0] = uint32_t(lo);
        nodeRange[2 * i + 1] = uint32_t(hi);
    }
    StoreBox(boxes + 6 * size_t(i), RangeBox(lv, uint32_t(lo), uint32_t(hi)));
}

// ---------------------------------------------------------------------------
// ValidateBinaryTree on the device, one thread per node: a node's children
// split its range at one point and name it as their parent.  With the root
// over all leaves that is the whole tree: a node has one stored parent, so
// nothing is reached twice, and a walk from the root splits n positions into
// single leaves, which takes all n - 1 nodes.
// ---------------------------------------------------------------------------
__global__ void __launch_bounds__(kTPB)
KCValidate(const uint32_t* __restrict__ nodes, const uint32_t* __restrict__ range,
           const uint32_t* __restrict__ leafOrder, uint32_t n, uint32_t* __restrict__ bad)
{
    const uint32_t v = blockIdx.x * blockDim.x + threadIdx.x;
    if(v >= n - 1u) return;
    const uint32_t lo = range[2 * size_t(v)], hi = range[2 * size_t(v) + 1];
    bool ok = lo < hi && hi < n && (v != 0u || (lo == 0u && hi == n - 1u));
    uint32_t mid = lo;
    for(uint32_t side = 0; side < 2 && ok; side++)
    {
        const uint32_t c = nodes[size_t(v) * 3 + side];
        const uint32_t first = side ? mid + 1u : lo;
        if(c & kLeafFlag)
        {
            ok = (!side || first == hi) && c == (kLeafFlag | leafOrder[first]);
            mid = first;
        }
        else
        {
            ok = c != 0u && c < n - 1u && nodes[size_t(c) * 3 + 2] == v && range[2 * size_t(c)] == first;
            mid = ok ? range[2 * size_t(c) + 1] : 0u;
            ok = ok && (side ? mid == hi : mid < hi);
        }
    }
    if(!ok) *bad = 1u;
}

__global__ void __launch_bounds__(kTPB) KCIota(uint32_t* __restrict__ out, uint32_t n)
{
    uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if(i < n) out[i] = i;
}

// ---------------------------------------------------------------------------
// Host-side launchers
// ---------------------------------------------------------------------------
int LaunchIota(uint32_t* dOut, uint32_t n, hipStream_t s)
{
    if(n == 0) return MRAY_OK;
    KCIota<<<DivUp(n, kTPB), kTPB, 0, s>>>(dOut, n);
    MRAY_HIP_CHECK(hipGetLastError());
    return MRAY_OK;
}

int LaunchPrimCentersAabbs(const float* dPos, const uint32_t* dIdx, uint32_t n, float* dCenters,
                           float* dAabbs, hipStream_t s)
{
    if(n == 0) return MRAY_OK;
    KCPrimCentersAabbs<<<DivUp(n, kTPB), kTPB, 0, s>>>(dPos, dIdx, n, dCenters, dAabbs);
    MRAY_HIP_CHECK(hipGetLastError());
    return MRAY_OK;
}

int LaunchReduceAabb(const float* dAabbs, uint32_t n, float* dOut, float* dPartial, hipStream_t s)
{
    uint32_t blocks = std::min<uint32_t>(kReduceBlocks, std::max<uint32_t>(1u, DivUp(n, kTPB)));
    KCReduceAabbPartial<<<blocks, kTPB, 0, s>>>(dAabbs, n, dPartial);
    MRAY_HIP_CHECK(hipGetLastError());
    KCReduceAabbPartial<<<1, kTPB, 0, s>>>(dPartial, blocks, dOut);
    MRAY_HIP_CHECK(hipGetLastError());
    return MRAY_OK;
}

size_t ReduceAabbTempBytes() { return size_t(kReduceBlocks) * 6 * sizeof(float); }

int LaunchMorton63(const float* dCenters, uint32_t n, const float* dBox, uint64_t* dCodes,
                   hipStream_t s)
{
    if(n == 0) return MRAY_OK;
    KCMorton63<<<DivUp(n, kTPB), kTPB, 0, s>>>(dCenters, n, dBox, dCodes);
    MRAY_HIP_CHECK(hipGetLastError());
    return MRAY_OK;
}

int LaunchMorton30(const float* dCenters, uint32_t n, const float* dBox, uint32_t* dCodes,
                   hipStream_t s)
{
    if(n == 0) return MRAY_OK;
    KCMorton30<<<DivUp(n, kTPB), kTPB, 0, s>>>(dCenters, n, dBox, dCodes);
    MRAY_HIP_CHECK(hipGetLastError());
    return MRAY_OK;
}

// Temporary area: tile histograms, digit totals, then the other half of the
// ping-pong pair.
static constexpr size_t RsHistBytes(uint32_t n)
{
    const size_t tiles = (size_t(n) + RsTile(n) - 1) / RsTile(n);
    return ((256u * (tiles ? tiles : 1u) + 256u) * sizeof(uint32_t) + 255) / 256 * 256;
}

// What a sort of n pairs uses.
static constexpr size_t RsNeed(size_t histBytes, uint32_t n)
{
    return histBytes + size_t(n) * (sizeof(uint64_t) + sizeof(uint32_t)) + 256;
}

// A workspace for n pairs serves every smaller count too: where tiles grow,
// the count just below has more histogram rows.
static constexpr size_t RsHistBytesUpTo(uint32_t n)
{
    size_t b = RsHistBytes(n);
    if(n >= kRsMidFrom) b = std::max(b, RsHistBytes(kRsMidFrom - 1u));
    if(n >= kRsLargeFrom) b = std::max(b, RsHistBytes(kRsLargeFrom - 1u));
    return b;
}
size_t RadixSortTempBytes(uint32_t n) { return RsNeed(RsHistBytesUpTo(n), n); }

template<uint32_t R>
static void LaunchRadixPass(const uint64_t* srcK, const uint32_t* srcV, uint64_t* dstK, uint32_t* dstV,
                            uint32_t n, uint32_t shift, uint32_t* hist, hipStream_t s)
{
    const uint32_t tiles = DivUp(n, kRsThreads * R);
    uint32_t* total = hist + size_t(256) * tiles;
    KCRadixHist<R><<<tiles, kRsThreads, 0, s>>>(srcK, n, shift, tiles, hist);
    KCRadixScan<<<256, kRsThreads, 0, s>>>(hist, tiles, total);
    KCRadixScatter<R><<<tiles, kRsThreads, 0, s>>>(srcK, srcV, dstK, dstV, n, shift, tiles, hist, total);
}

int LaunchRadixSort(uint64_t* dKeys, uint32_t* dVals, uint32_t n, void* dTemp, size_t tempBytes,
                    hipStream_t s)
{
    if(n <= 1) return MRAY_OK;
    if(tempBytes < RsNeed(RsHistBytes(n), n))
    {
        SetError("radix sort: temporary buffer too small");
        return MRAY_ERR_INVALID;
    }
    if(n <= kRsOneMax)
    {
        if(n <= kRsOneThreads * 4u) KCRadixSortOneGroup<4><<<1, kRsOneThreads, 0, s>>>(dKeys, dVals, n);
        else KCRadixSortOneGroup<12><<<1, kRsOneThreads, 0, s>>>(dKeys, dVals, n);
        MRAY_HIP_CHECK(hipGetLastError());
        return MRAY_OK;
    }
    char* t = static_cast<char*>(dTemp);
    uint32_t* hist = reinterpret_cast<uint32_t*>(t);
    uint64_t* altK = reinterpret_cast<uint64_t*>(t + RsHistBytes(n));
    uint32_t* altV = reinterpret_cast<uint32_t*>(altK + n);
    uint64_t* srcK = dKeys;
    uint32_t* srcV = dVals;
    uint64_t* dstK = altK;
    uint32_t* dstV = altV;
    for(uint32_t pass = 0; pass < 8; pass++)
    {
        switch(RsRounds(n))
        {
            case 4: LaunchRadixPass<4>(srcK, srcV, dstK, dstV, n, pass * 8u, hist, s); break;
            case 8: LaunchRadixPass<8>(srcK, srcV, dstK, dstV, n, pass * 8u, hist, s); break;
            default: LaunchRadixPass<12>(srcK, srcV, dstK, dstV, n, pass * 8u, hist, s); break;
        }
        MRAY_HIP_CHECK(hipGetLastError());
        std::swap(srcK, dstK);
        std::swap(srcV, dstV);
    }
    // 8 passes: the result is back in the caller's buffers
    return MRAY_OK;
}

// ---------------------------------------------------------------------------
// Allocation-free sort (mray_radix_sort_u64_u32_noalloc): the same passes over
// a scratch area that lives in the code object, one copy per GPU, held until
// the process ends, large enough for every count up to kNoAllocSortMax.
// ---------------------------------------------------------------------------
constexpr uint32_t kNoAllocSortMax = MRAY_NOALLOC_SORT_MAX;
static_assert(kNoAllocSortMax == (1u << 20), "scratch size is stated as 2^20 pairs");
constexpr size_t kNoAllocSortBytes = RsNeed(RsHistBytesUpTo(kNoAllocSortMax), kNoAllocSortMax);
static __device__ __align__(256) unsigned char scratch[kNoAllocSortBytes];

namespace
{
constexpr int kMaxDevices = 64;
std::mutex gScratchLock;
void* gScratchPtr[kMaxDevices] = {};
}

// The device address of `scratch` on the current GPU, looked up once per GPU
// (the array's name is only a host-side handle; kernels need this address).
static int ScratchOnCurrentDevice(void** out)
{
    int dev = 0;
    MRAY_HIP_CHECK(hipGetDevice(&dev));
    if(dev < 0 || dev >= kMaxDevices)
    {
        SetError("radix sort (no-alloc): device index out of range");
        return MRAY_ERR_INVALID;
    }
    std::lock_guard<std::mutex> g(gScratchLock);
    if(!gScratchPtr[dev])
    {
        void* p = nullptr;
        MRAY_HIP_CHECK(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
        if(!p)
        {
            SetError("radix sort (no-alloc): scratch symbol has no device address");
            return MRAY_ERR_HIP;
        }
        gScratchPtr[dev] = p;
    }
    *out = gScratchPtr[dev];
    return MRAY_OK;
}

size_t LbvhTempBytes(uint32_t n)
{
    // box levels (about 43 B per leaf), aligned to 16 B inside the caller's area
    return BoxLevelEntries(std::max(n, 1u), nullptr) * sizeof(LevelBox) + 256;
}

int LaunchLbvhBuild(const uint64_t* dSortedCodes, const uint32_t* dLeafOrder,
                    const float* dLeafAabbs, uint32_t n, uint32_t* dNodes, float* dBoxes,
                    uint32_t* dNodeRange, void* dTemp, size_t tempBytes, hipStream_t s,
                    uint32_t strictTie)
{
    if(n == 0) return MRAY_OK;
    if(tempBytes < LbvhTempBytes(n))
    {
        SetError("lbvh build: temporary buffer too small");
        return MRAY_ERR_INVALID;
    }
    BoxLevels lv{};
    lv.base = reinterpret_cast<LevelBox*>((reinterpret_cast<uintptr_t>(dTemp) + 15u) & ~uintptr_t(15));
    BoxLevelEntries(n, &lv);
    KCLeafLevels<<<DivUp(n, kLevelTPB), kLevelTPB, 0, s>>>(dLeafOrder, dLeafAabbs, n, lv, dNodes);
    MRAY_HIP_CHECK(hipGetLastError());
    if(lv.levels > kLevelsPerBlock + 1u)
    {
        KCTopLevels<<<1, 1024, 0, s>>>(lv);
        MRAY_HIP_CHECK(hipGetLastError());
    }
    KCKarras<<<DivUp(std::max(n - 1, 1u), kTPB), kTPB, 0, s>>>(dSortedCodes, dLeafOrder, int32_t(n), dNodes,
                                                               dNodeRange, lv, dBoxes, strictTie);
    MRAY_HIP_CHECK(hipGetLastError());
    return MRAY_OK;
}

int ValidateTreeDevice(const uint32_t* dNodes, const uint32_t* dRange, const uint32_t* dLeafOrder,
                       uint32_t n, uint32_t* dFlag, hipStream_t s, bool* ok)
{
    *ok = false;
    uint32_t bad = 1u;
    if(n == 1)
    {
        uint32_t node0 = 0;
        MRAY_HIP_CHECK(hipMemcpyAsync(&node0, dNodes, 4, hipMemcpyDeviceToHost, s));
        MRAY_HIP_CHECK(hipStreamSynchronize(s));
        bad = (node0 != (kLeafFlag | 0u)) ? 1u : 0u;
    }
    else
    {
        MRAY_HIP_CHECK(hipMemsetAsync(dFlag, 0, 4, s));
        KCValidate<<<DivUp(n - 1u, kTPB), kTPB, 0, s>>>(dNodes, dRange, dLeafOrder, n, dFlag);
        MRAY_HIP_CHECK(hipGetLastError());
        MRAY_HIP_CHECK(hipMemcpyAsync(&bad, dFlag, 4, hipMemcpyDeviceToHost, s));
        MRAY_HIP_CHECK(hipStreamSynchronize(s));
    }
    *ok = bad == 0u;
    return MRAY_OK;
}

} // namespace mray

using namespace mray;

extern "C" int mray_radix_sort_u64_u32_noalloc(uint64_t* dKeys, uint32_t* dValues, uint32_t count,
                                                void* stream)
{
    if(count > kNoAllocSortMax)
    {
        SetError("radix sort (no-alloc): " + std::to_string(count) + " pairs exceed the maximum of " +
                 std::to_string(kNoAllocSortMax));
        return MRAY_ERR_INVALID;
    }
    if(count > 1 && (!dKeys || !dValues))
    {
        SetError("radix sort (no-alloc): NULL keys or values");
        return MRAY_ERR_INVALID;
    }
    if(count <= 1) return MRAY_OK;
    void* tmp = nullptr;
    MRAY_TRY(ScratchOnCurrentDevice(&tmp));
    return LaunchRadixSort(dKeys, dValues, count, tmp, kNoAllocSortBytes,
                           static_cast<hipStream_t>(stream));
}

