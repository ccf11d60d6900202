// Neural radiance cache on gfx950: multiresolution hash encoding + 64-wide
// fully fused MLP on bf16 MFMA (fp32 accumulation), trained online with Adam.
//
// No reference counterpart (the reference only keeps an irradiance hash grid,
// Tracer/HashGrid.h:17-476); the methods are the published ones: hash
// encoding of Mueller et al. 2022 (Instant NGP), one-blob encoding of Mueller
// et al. 2019, network and relative L2 loss of Mueller et al. 2021 (Real-time
// Neural Radiance Caching).
//
// Query record (11 floats): position in [0,1]^3 (scene box), direction and
// normal as (theta, phi) in [0,1]^2, roughness in [0,1], albedo RGB.
// Network input (64): 16 levels x 2 hash features, one-blob(4) of the five
// scalars, albedo, a constant 1, zero padding.  Six 64x64 layers (the output
// layer's columns 3..63 stay zero), ReLU after the first five.
//
// Kernels (one wave = 32 samples; the MFMA is gfx950's v_mfma_f32_32x32x16_bf16,
// 16 k per instruction, with weights as A and samples as columns of B, so a
// lane's accumulators are consecutive features of its own sample: packed to
// bf16 they are the next layer's B operand, and activations never leave
// registers):
//   KNrcInfer      encode + 6 layers for queries, weights in LDS
//   KNrcTrain      encode, forward, loss gradient and the data gradients of
//                  every layer in one pass; stores each layer's input and
//                  output gradient transposed (samples contiguous) and the
//                  gradient of the grid features
//   KNrcWgrad      dW = X^T dZ, one workgroup per 16 x 16 tile over all
//                  samples, no atomics; with Adam fused in a training step
//   KNrcGridOwner  grid gradient: a workgroup owns a table segment in LDS and
//                  scans the batch for corners inside it; with Adam fused in
//                  a training step
//   KNrcGridBwd    grid gradient by global atomics (tables too large or
//                  batches too small for the scan)
//   KNrcAdam*      Adam on fp32 masters as a separate pass (mray_nrc_adam)
#include "common.h"
#include "scene.h"

#include <hip/hip_fp16.h>

#include <cmath>
#include <cstring>
#include <map>
#include <mutex>
#include <random>
#include <vector>

namespace mray
{

typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
typedef float v16f __attribute__((ext_vector_type(16)));

constexpr uint32_t kNrcLayers = 6;
constexpr uint32_t kW = 64;                  // width of every layer
constexpr uint32_t kNrcFeat = 2;
constexpr uint32_t kNrcMaxLevels = 16;
constexpr uint32_t kInferTPB = 512;          // 8 waves: 256 queries per block and round
constexpr uint32_t kEncodeTPB = 256;
constexpr uint32_t kSplitChunk = 1u << 19;   // queries encoded at a time (32 MiB of features)
constexpr uint32_t kLayerParams = kW * kW;
constexpr uint32_t kMlpParams = kNrcLayers * kLayerParams;
// kernel kinds timed by mray_nrc_kernel_times: inference forward, training
// forward, backward (data gradients), weight gradients, grid scatter, Adam.
// A fused kernel counts under the first of its parts: forward and data
// gradients as training forward, and in a training step Adam with the
// gradients it applies.
constexpr uint32_t kNrcKernelKinds = 6;

__device__ __forceinline__ uint16_t F2Bf(float f)
{
    uint32_t u = __float_as_uint(f);
    u += 0x7FFFu + ((u >> 16) & 1u);         // round to nearest even
    return uint16_t(u >> 16);
}

struct NrcView
{
    const uint16_t* wT;       // bf16, fragment order: forward operand (rows n)
    const uint16_t* wK;       // bf16, fragment order: backward operand (rows k)
    const __half* grid;       // [L][T][2]
    float scale[kNrcMaxLevels];
    uint32_t my[kNrcMaxLevels];      // index multipliers of y and z: the level's
    uint32_t mz[kNrcMaxLevels];      // resolution and its square, or the hash primes
    uint32_t dense[kNrcMaxLevels];
    uint32_t levels;
    uint32_t log2T;
};

// ---- operand layout ----------------------------------------------------------
// v_mfma_f32_32x32x16_bf16 D = A B: lane (r, h) = (l mod 32, l / 32) supplies
// row r of A and column r of B over eight of the step's 16 k, and receives
// column r of D, rows 8 (e / 4) + 4 h + (e mod 4) for e = 0..15.  The k order
// inside a step is free as long as A and B agree: slot j of half h in step kt
// is k = 16 kt + 8 (j / 4) + 4 h + (j mod 4), so D's rows, packed in pairs,
// are the next product's B operand in the lane that holds them.
// Element (row, k) of layer l's A operand in fragment order
// [layer][32-row tile][step][lane][8]: a lane's operand is 16 contiguous
// bytes and a wave's 1 KiB, conflict-free in LDS and coalesced from memory.
__host__ __device__ constexpr uint32_t FragIndex(uint32_t l, uint32_t row, uint32_t k)
{
    const uint32_t c = k & 15u, j = 4u * (c >> 3) + (c & 3u), h = (c >> 2) & 1u;
    return (((l * 2u + (row >> 5)) * 4u + (k >> 4)) * 64u + (row & 31u) + 32u * h) * 8u + j;
}
constexpr uint32_t kFragLayer = 2u * 4u * 64u;   // uint4 words of one layer

__device__ __forceinline__ uint32_t PackBf(float a, float b)
{
    typedef __bf16 v2bf __attribute__((ext_vector_type(2)));
    const v2bf v = {__bf16(a), __bf16(b)};       // v_cvt_pk_bf16_f32, nearest even
    return __builtin_bit_cast(uint32_t, v);
}

// B operand of one wave: 64 features of the lane's sample, word 4 kt + i =
// slots 2i, 2i + 1 of step kt.
struct XRow
{
    uint32_t u[32 / 2];
};

__device__ __forceinline__ v8bf StepOf(const XRow& x, uint32_t kt)
{
    const uint4 v = make_uint4(x.u[4 * kt], x.u[4 * kt + 1], x.u[4 * kt + 2], x.u[4 * kt + 3]);
    return __builtin_bit_cast(v8bf, v);
}

// One layer's A operand in registers.
struct Frags
{
    uint4 f[8];
};
__device__ __forceinline__ Frags LoadFrags(const uint4* __restrict__ w)
{
    Frags a;
    #pragma unroll
    for(uint32_t i = 0; i < 8; i++) a.f[i] = w[i * 64u + (threadIdx.x & 63u)];
    return a;
}
template<uint32_t TILES, uint32_t STEPS>
__device__ __forceinline__ void LayerProduct(const Frags& w, const XRow& x, v16f (&acc)[2])
{
    acc[0] = v16f{0};
    acc[1] = v16f{0};
    #pragma unroll
    for(uint32_t kt = 0; kt < STEPS; kt++)
        #pragma unroll
        for(uint32_t t = 0; t < TILES; t++)
            acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(v8bf, w.f[t * 4u + kt]),
                                                             StepOf(x, kt), acc[t], 0, 0, 0);
}

// acc[t] = rows 32 t.. of one layer's A times x, over the first `steps` k steps.
template<uint32_t TILES, uint32_t STEPS>
__device__ __forceinline__ void LayerProduct(const uint4* __restrict__ w, const XRow& x, v16f (&acc)[2])
{
    const uint32_t lane = threadIdx.x & 63u;
    acc[0] = v16f{0};
    acc[1] = v16f{0};
    #pragma unroll
    for(uint32_t kt = 0; kt < STEPS; kt++)
    {
        const v8bf b = StepOf(x, kt);
        #pragma unroll
        for(uint32_t t = 0; t < TILES; t++)
        {
            const v8bf a = __builtin_bit_cast(v8bf, w[(t * 4u + kt) * 64u + lane]);
            acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, acc[t], 0, 0, 0);
        }
    }
}

__device__ __forceinline__ XRow ReluPack(const v16f (&acc)[2])
{
    XRow x;
    #pragma unroll
    for(uint32_t t = 0; t < 2; t++)
        #pragma unroll
        for(uint32_t i = 0; i < 8; i++)
            x.u[8 * t + i] = PackBf(MaxF(acc[t][2 * i], 0.0f), MaxF(acc[t][2 * i + 1], 0.0f));
    return x;
}

// ---- encoding --------------------------------------------------------------
__device__ __forceinline__ uint32_t GridIndex(uint32_t dense, uint32_t mask, uint32_t x, uint32_t y, uint32_t z)
{
    return dense ? x + y + z : ((x ^ y ^ z) & mask);
}

// Cell and fraction of a position on one level; iy and iz already multiplied.
struct Cell
{
    uint32_t x, y, z;
    float fx, fy, fz;
};
__device__ __forceinline__ Cell LevelCell(const float* pos, float scale, uint32_t my, uint32_t mz)
{
    const float px = pos[0] * scale + 0.5f, py = pos[1] * scale + 0.5f, pz = pos[2] * scale + 0.5f;
    const float gx = floorf(px), gy = floorf(py), gz = floorf(pz);
    return {uint32_t(gx), uint32_t(gy) * my, uint32_t(gz) * mz, px - gx, py - gy, pz - gz};
}
__device__ __forceinline__ float CornerWeight(const Cell& c, uint32_t k)
{
    float w = (k & 1u) ? c.fx : 1.0f - c.fx;
    w = w * ((k & 2u) ? c.fy : 1.0f - c.fy);
    return w * ((k & 4u) ? c.fz : 1.0f - c.fz);
}

__device__ __forceinline__ float OneBlob(float s, uint32_t j)
{
    float c = (float(j) + 0.5f) * 0.25f;
    float d = s - c;
    return expf(-d * d * 8.0f);              // sigma = 1/4
}

__device__ __forceinline__ void RecordPos(const float* __restrict__ rec, float pos[3])
{
    for(int k = 0; k < 3; k++) pos[k] = ClampF(rec[k], 0.0f, 1.0f);
}

// Interpolated features of one level, corners summed in order.  The two corners
// along x are one entry apart in the low index bits, so an aligned 16-byte
// load of four entries brings both unless x mod 4 is 3: 5 gathers per 4 pairs
// instead of 8 (QUADS; otherwise 8 single gathers).
template<bool QUADS>
__device__ __forceinline__ uint32_t LevelFeatures(const uint32_t* __restrict__ table, const float pos[3],
                                                  float scale, uint32_t my, uint32_t mz, uint32_t dense,
                                                  uint32_t mask)
{
    const Cell c = LevelCell(pos, scale, my, mz);
    uint4 quad[4];
    uint32_t i0[4], i1[4], e0[4], e1[4];
    #pragma unroll
    for(uint32_t q = 0; q < 4; q++)
    {
        const uint32_t y = c.y + ((q & 1u) ? my : 0u), z = c.z + ((q & 2u) ? mz : 0u);
        i0[q] = GridIndex(dense, mask, c.x, y, z);
        i1[q] = GridIndex(dense, mask, c.x + 1u, y, z);
        if constexpr(QUADS)
        {
            quad[q] = *reinterpret_cast<const uint4*>(table + (i0[q] & ~3u));
            e1[q] = 0u;
            if((i0[q] ^ i1[q]) > 3u) e1[q] = table[i1[q]];
        }
        else
        {
            e0[q] = table[i0[q]];
            e1[q] = table[i1[q]];
        }
    }
    float f0 = 0.0f, f1 = 0.0f;
    #pragma unroll
    for(uint32_t q = 0; q < 4; q++)
    {
        auto pick = [&](uint32_t i)
        {
            const uint32_t lo = (i & 2u) ? quad[q].z : quad[q].x, hi = (i & 2u) ? quad[q].w : quad[q].y;
            return (i & 1u) ? hi : lo;
        };
        if constexpr(QUADS)
        {
            e0[q] = pick(i0[q]);
            if((i0[q] ^ i1[q]) <= 3u) e1[q] = pick(i1[q]);
        }
        #pragma unroll
        for(uint32_t k = 0; k < 2; k++)
        {
            const float w = CornerWeight(c, 2u * q + k);
            const float2 g = __half22float2(__builtin_bit_cast(__half2, k ? e1[q] : e0[q]));
            f0 += w * g.x;
            f1 += w * g.y;
        }
    }
    return PackBf(f0, f1);
}

// Words 8..13 of half h's operand: one-blobs h and 2 + h, then its share of
// the last 16 columns (words 14 and 15 are zero).
__device__ __forceinline__ void EncodeTail(const float* __restrict__ rec, bool hi, XRow& x)
{
    const float qa = hi ? rec[4] : rec[3], qb = hi ? rec[6] : rec[5], r7 = rec[7];
    x.u[8] = PackBf(OneBlob(qa, 0), OneBlob(qa, 1));
    x.u[9] = PackBf(OneBlob(qa, 2), OneBlob(qa, 3));
    x.u[10] = PackBf(OneBlob(qb, 0), OneBlob(qb, 1));
    x.u[11] = PackBf(OneBlob(qb, 2), OneBlob(qb, 3));
    x.u[12] = hi ? PackBf(rec[8], rec[9]) : PackBf(OneBlob(r7, 0), OneBlob(r7, 1));
    x.u[13] = hi ? PackBf(rec[10], 1.0f) : PackBf(OneBlob(r7, 2), OneBlob(r7, 3));
    x.u[14] = 0u;
    x.u[15] = 0u;
}

// Word m of an operand holds level LevelOfWord(m) in the lower half of the
// wave and that level plus 2 in the upper.
__device__ constexpr uint32_t LevelOfWord(uint32_t m) { return 4u * (m >> 1) + (m & 1u); }

// Operand of sample (lane mod 32), two lanes per sample: each takes the 8
// levels its words hold.  Both halves run one instruction stream: a step's
// two levels' constants are picked per half from scalar registers.
// QUADS = false issues 8 independent gathers per level and has no branch, so
// that the gathers of several levels are in flight together: for kernels with
// few waves, where latency counts and not the gather rate.
template<bool QUADS>
__device__ __forceinline__ XRow EncodePair(const NrcView& v, const float* __restrict__ rec, const float pos[3])
{
    const bool hi = (threadIdx.x & 32u) != 0u;
    const uint32_t mask = (1u << v.log2T) - 1u;
    const uint32_t* __restrict__ grid = reinterpret_cast<const uint32_t*>(v.grid);
    XRow x;
    #pragma unroll
    for(uint32_t m = 0; m < 8; m++)
    {
        // levels past the last read the last one and are dropped
        const uint32_t la = LevelOfWord(m), lb = la + 2u;
        x.u[m] = 0u;
        if(QUADS && la >= v.levels) continue;
        const uint32_t ra = min(la, v.levels - 1u), rb = min(lb, v.levels - 1u);
        const uint32_t f = LevelFeatures<QUADS>(grid + (size_t(hi ? rb : ra) << v.log2T), pos,
                                                hi ? v.scale[rb] : v.scale[ra], hi ? v.my[rb] : v.my[ra],
                                                hi ? v.mz[rb] : v.mz[ra], hi ? v.dense[rb] : v.dense[ra], mask);
        x.u[m] = ((hi ? lb : la) < v.levels) ? f : 0u;
    }
    EncodeTail(rec, hi, x);
    return x;
}

// ---- inference ---------------------------------------------------------------
// A tile's six layers and its three outputs.
__device__ __forceinline__ void InferLayers(const uint4* sW, XRow& x, float* __restrict__ out, size_t s, size_t n)
{
    v16f acc[2];
    #pragma unroll 1
    for(uint32_t l = 0; l + 1u < kNrcLayers; l++)
    {
        LayerProduct<2, 4>(sW + l * kFragLayer, x, acc);
        x = ReluPack(acc);
    }
    LayerProduct<1, 4>(sW + (kNrcLayers - 1u) * kFragLayer, x, acc);
    if((threadIdx.x & 32u) == 0u && s < n)
        for(uint32_t c = 0; c < 3; c++) out[s * 3u + c] = acc[0][c];
}

__device__ __forceinline__ void StageWeights(const NrcView& v, uint4* sW)
{
    for(uint32_t i = threadIdx.x; i < kNrcLayers * kFragLayer; i += kInferTPB)
        sW[i] = reinterpret_cast<const uint4*>(v.wT)[i];
    __syncthreads();
}

// The one-kernel form, for a count that only the device knows (the renderer's
// query queues, mostly empty) and for captured calls: persistent waves over
// 32-query tiles, weights staged once per block (48 KiB in fragment order).
// Bound by the latency of the grid gathers.
__global__ void __launch_bounds__(kInferTPB)
KNrcInfer(NrcView v, const float* __restrict__ rec, const uint32_t* __restrict__ dCount, uint32_t count,
          float* __restrict__ out)
{
    __shared__ uint4 sW[kNrcLayers * kFragLayer];
    const uint32_t n = dCount ? *dCount : count;
    constexpr uint32_t kWaves = kInferTPB / 64u;
    // a block without a tile (few or no queries this bounce) skips the
    // weight staging: the test is uniform over the block
    if(size_t(blockIdx.x) * kWaves * 32u >= n) return;
    StageWeights(v, sW);
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    for(size_t tile = blockIdx.x * kWaves + wave; tile * 32u < n; tile += gridDim.x * kWaves)
    {
        // lanes past the last query repeat it and write nothing
        const size_t s = tile * 32u + (lane & 31u);
        const float* r = rec + min(s, size_t(n) - 1u) * 11u;
        float pos[3];
        RecordPos(r, pos);
        XRow x = EncodePair<true>(v, r, pos);
        InferLayers(sW, x, out, s, n);
    }
}

// A count known on the host: encoding by level first, one lane per query and
// level.  One level's table (2 MiB at 2^19 entries) fits an XCD's 4 MiB L2, all
// of them (22 MiB) do not, and waves that walk the levels on their own spread
// over all of them (33 M of 84 M L2 reads missed per 10^6 queries, now 5.6 of
// 61).  Workgroups go round-robin over the 8 XCDs, so workgroup 8 j + x is the
// j-th of XCD x: it first takes its own hashed levels for every query, then an
// eighth of the queries for each remaining level.
// 16 levels of 2^19 entries: 10^6 queries 643 -> 290 us of encoding (L2 serves
// 211 reads/ns, near its 16 channels per XCD a clock) + 70 us of layers; 4096
// queries 41 -> 26 us, because the lanes are 16 times as many.  Chunks of 2^18
// and 2^17 queries cost 9 and 22 % more.
struct EncodePlan
{
    uint32_t own;                            // hashed levels per XCD
    uint32_t shared;                         // levels shared by all XCDs
    uint32_t ownLevel[kNrcMaxLevels];        // [own][8]
    uint32_t sharedLevel[kNrcMaxLevels];
};
__global__ void __launch_bounds__(kEncodeTPB)
KNrcEncode(NrcView v, const float* __restrict__ rec, uint32_t n, EncodePlan plan, uint32_t* __restrict__ feat)
{
    const uint32_t blocks = (n + kEncodeTPB - 1u) / kEncodeTPB, eighth = (blocks + 7u) / 8u;
    const uint32_t xcd = blockIdx.x & 7u, j = blockIdx.x >> 3;
    uint32_t l, b;
    if(j < plan.own * blocks)
    {
        l = plan.ownLevel[(j / blocks) * 8u + xcd];
        b = j % blocks;
    }
    else
    {
        const uint32_t i = j - plan.own * blocks;
        l = plan.sharedLevel[i / eighth];
        b = (i % eighth) * 8u + xcd;
    }
    const uint32_t s = b * kEncodeTPB + threadIdx.x;
    if(s >= n) return;
    float pos[3];
    RecordPos(rec + size_t(s) * 11u, pos);
    feat[size_t(l) * n + s] = LevelFeatures<true>(reinterpret_cast<const uint32_t*>(v.grid) + (size_t(l) << v.log2T), pos,
                                                  v.scale[l], v.my[l], v.mz[l], v.dense[l], (1u << v.log2T) - 1u);
}

// The layers over encoded queries.
__global__ void __launch_bounds__(kInferTPB)
KNrcInferEncoded(NrcView v, const float* __restrict__ rec, const uint32_t* __restrict__ feat, uint32_t n,
                 float* __restrict__ out)
{
    __shared__ uint4 sW[kNrcLayers * kFragLayer];
    constexpr uint32_t kWaves = kInferTPB / 64u;
    StageWeights(v, sW);
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    const bool hi = (lane & 32u) != 0u;
    for(size_t tile = blockIdx.x * kWaves + wave; tile * 32u < n; tile += gridDim.x * kWaves)
    {
        const size_t s = tile * 32u + (lane & 31u), at = min(s, size_t(n) - 1u);
        XRow x;
        #pragma unroll
        for(uint32_t m = 0; m < 8; m++)
        {
            const uint32_t l = LevelOfWord(m) + (hi ? 2u : 0u);
            x.u[m] = (l < v.levels) ? feat[size_t(l) * n + at] : 0u;
        }
        EncodeTail(rec + at * 11u, hi, x);
        InferLayers(sW, x, out, s, n);
    }
}

// ---- training: forward and data gradients -----------------------------------
// What a training call leaves for later ones, in device memory: a captured call
// runs again at each replay, which the host does not see.
struct NrcState
{
    uint32_t pending;  // gradients of a backward pass that no Adam step has applied
    uint32_t apply;    // of the running fused step: it applies pending gradients
    uint32_t tiles;    // tiles of the last batch
};
struct NrcTrainBuf
{
    NrcState* state;
    uint32_t* x;       // [6][B/32][64 features][32 samples] bf16 layer inputs
    uint32_t* dz;      // the same for the gradients of the layer outputs
    float2* dx0;       // [16 levels][B] gradient of the grid features
    float* pos;        // [3][B] clamped positions
    float* loss;       // [B/32] each tile's part of the loss
};

// Stores packed features (word q of XRow: q and q + 1 of the lane's sample)
// with the samples contiguous: neighbouring lanes swap a feature, so each lane
// writes two samples of one feature.
__device__ __forceinline__ void StoreTransposed(uint32_t* __restrict__ rows, const XRow& x, uint32_t words)
{
    const uint32_t lane = threadIdx.x & 63u, h = lane >> 5, s = lane & 31u, odd = s & 1u;
    const uint32_t sel = odd ? 0x03020706u : 0x05040100u;
    #pragma unroll
    for(uint32_t q = 0; q < 16; q++)
    {
        if(q >= words) break;
        const uint32_t i = q & 7u;
        const uint32_t f = 32u * (q >> 3) + 8u * (i >> 1) + 4u * h + 2u * (i & 1u) + odd;
        const uint32_t other = uint32_t(__builtin_amdgcn_update_dpp(0, int(x.u[q]), 0xB1, 0xF, 0xF, true));
        rows[f * 16u + (s >> 1)] = __builtin_amdgcn_perm(other, x.u[q], sel);
    }
}

// One wave per 32 samples, everything in registers; weights come straight from
// L2 in fragment order (a training batch is about two waves per CU, so staging
// them in LDS would cost more than the products): batch 16384: 23 us,
// from 53 + 55 us as two LDS-staged kernels.
__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(1, 2)))
KNrcTrain(NrcView v, const float* __restrict__ rec, const float* __restrict__ target, NrcTrainBuf tb,
          uint32_t batch, uint32_t step)
{
    const uint32_t lane = threadIdx.x & 63u, tiles = batch / 32u, tile = blockIdx.x;
    if(tile == 0u && lane == 0u)
    {
        // a fused step (step = 1) takes over what is pending, a backward pass adds to it
        tb.state->apply = tb.state->pending;
        tb.state->pending = step ? 0u : 1u;
        tb.state->tiles = tiles;
    }
    const uint32_t s = tile * 32u + (lane & 31u);
    const float* r = rec + size_t(s) * 11u;
    const uint4* __restrict__ wT = reinterpret_cast<const uint4*>(v.wT);
    const uint4* __restrict__ wK = reinterpret_cast<const uint4*>(v.wK);
    float pos[3];
    RecordPos(r, pos);
    if(lane < 32u)
        for(uint32_t k = 0; k < 3; k++) tb.pos[size_t(k) * batch + s] = pos[k];
    auto rows = [&](uint32_t* base, uint32_t l) { return base + (size_t(l) * tiles + tile) * 64u * 16u; };
    XRow x[kNrcLayers];
    v16f acc[2];
    // each layer's weights are loaded while the layer before it is computed
    Frags w = LoadFrags(wT);
    x[0] = EncodePair<false>(v, r, pos);
    #pragma unroll
    for(uint32_t l = 0; l + 1u < kNrcLayers; l++)
    {
        const Frags next = LoadFrags(wT + (l + 1u) * kFragLayer);
        StoreTransposed(rows(tb.x, l), x[l], 16);
        LayerProduct<2, 4>(w, x[l], acc);
        x[l + 1] = ReluPack(acc);
        w = next;
    }
    {
        const Frags next = LoadFrags(wK + (kNrcLayers - 1u) * kFragLayer);
        StoreTransposed(rows(tb.x, kNrcLayers - 1u), x[kNrcLayers - 1], 16);
        LayerProduct<1, 4>(w, x[kNrcLayers - 1], acc);
        w = next;
    }
    // relative L2 loss and its gradient: outputs 0..2 sit in the lower half
    float loss = 0.0f, dy[3] = {0.0f, 0.0f, 0.0f};
    if(lane < 32u)
        for(uint32_t c = 0; c < 3; c++)
        {
            const float y = acc[0][c], d = y - target[size_t(s) * 3u + c], den = y * y + 0.01f;
            loss += d * d / den;
            dy[c] = 2.0f * d / den / float(batch * 3u);
        }
    for(uint32_t o = 32; o > 0; o >>= 1) loss += __shfl_down(loss, o);
    if(lane == 0) tb.loss[tile] = loss / float(batch * 3u);
    XRow g;
    for(uint32_t q = 0; q < 16; q++) g.u[q] = 0u;
    g.u[0] = PackBf(dy[0], dy[1]);
    g.u[1] = PackBf(dy[2], 0.0f);
    // the output layer's gradient has 3 rows; its weight tile reads 16
    StoreTransposed(rows(tb.dz, kNrcLayers - 1u), g, 4);
    #pragma unroll
    for(uint32_t l = kNrcLayers - 1u; l > 0u; l--)
    {
        // dX = W dZ, then the ReLU that produced X
        const Frags next = LoadFrags(wK + (l - 1u) * kFragLayer);
        if(l == kNrcLayers - 1u) LayerProduct<2, 1>(w, g, acc);
        else LayerProduct<2, 4>(w, g, acc);
        w = next;
        #pragma unroll
        for(uint32_t q = 0; q < 16; q++)
        {
            const uint32_t in = x[l].u[q], t = q >> 3, i = q & 7u;
            g.u[q] = PackBf((in & 0xFFFFu) ? acc[t][2 * i] : 0.0f, (in >> 16) ? acc[t][2 * i + 1] : 0.0f);
        }
        StoreTransposed(rows(tb.dz, l - 1u), g, 16);
    }
    // gradient of the 32 grid features: rows 2 level, 2 level + 1
    LayerProduct<1, 4>(w, g, acc);
    #pragma unroll
    for(uint32_t i = 0; i < 8; i++)
    {
        const uint32_t level = 4u * (i >> 1) + 2u * (lane >> 5) + (i & 1u);
        tb.dx0[size_t(level) * batch + s] = make_float2(acc[0][2 * i], acc[0][2 * i + 1]);
    }
}

// ---- grid gradients -----------------------------------------------------------
// One thread per (sample, level): the 16 atomics of a level's 8 corners.
__global__ void __launch_bounds__(256)
KNrcGridBwd(NrcView v, NrcTrainBuf tb, uint32_t batch, float* __restrict__ ggrad)
{
    const uint32_t s = blockIdx.x * blockDim.x + threadIdx.x, l = blockIdx.y;
    if(s >= batch) return;
    const float2 g = tb.dx0[size_t(l) * batch + s];
    if(g.x == 0.0f && g.y == 0.0f) return;
    const float pos[3] = {tb.pos[s], tb.pos[batch + s], tb.pos[2 * size_t(batch) + s]};
    const Cell c = LevelCell(pos, v.scale[l], v.my[l], v.mz[l]);
    float* gl = ggrad + (size_t(l) << v.log2T) * 2u;
    for(uint32_t k = 0; k < 8; k++)
    {
        const size_t i = GridIndex(v.dense[l], (1u << v.log2T) - 1u, c.x + (k & 1u),
                                   c.y + ((k & 2u) ? v.my[l] : 0u), c.z + ((k & 4u) ? v.mz[l] : 0u));
        const float w = CornerWeight(c, k);
        atomicAdd(gl + i * 2u, w * g.x);
        atomicAdd(gl + i * 2u + 1u, w * g.y);
    }
}

// ---- Adam ---------------------------------------------------------------------
struct AdamArgs
{
    float lr, b1, b2, eps, c1, c2;   // c1 = 1/(1-b1^t), c2 = 1/(1-b2^t)
};

__device__ __forceinline__ float AdamOne(float& p, float& m, float& vv, float& g, const AdamArgs& a)
{
    float gg = g;
    g = 0.0f;
    m = a.b1 * m + (1.0f - a.b1) * gg;
    vv = a.b2 * vv + (1.0f - a.b2) * gg * gg;
    float mh = m * a.c1, vh = vv * a.c2;
    p = p - a.lr * mh / (sqrtf(vh) + a.eps);
    return p;
}

// One MLP parameter's update: columns past the three outputs stay zero.
struct MlpAdam
{
    float* w;
    float* m;
    float* v;
    uint16_t* wT;
    uint16_t* wK;
};
__device__ __forceinline__ void StoreWeight(uint16_t* wT, uint16_t* wK, uint32_t l, uint32_t k, uint32_t n, float p)
{
    const uint16_t b = F2Bf(p);
    wT[FragIndex(l, n, k)] = b;
    wK[FragIndex(l, k, n)] = b;
}
__device__ __forceinline__ void AdamWeight(const MlpAdam& u, uint32_t i, float g, const AdamArgs& a)
{
    const uint32_t l = i / kLayerParams, e = i % kLayerParams, k = e / kW, n = e % kW;
    const bool unused = l == kNrcLayers - 1u && n >= 3u;
    float p = u.w[i], m = u.m[i], v = u.v[i];
    if(unused) { p = 0.0f; g = 0.0f; }
    AdamOne(p, m, v, g, a);
    if(unused) p = 0.0f;
    u.w[i] = p; u.m[i] = m; u.v[i] = v;
    StoreWeight(u.wT, u.wK, l, k, n, p);
}

__global__ void __launch_bounds__(256)
KNrcAdamMlp(MlpAdam u, float* __restrict__ g, AdamArgs a, NrcState* __restrict__ state)
{
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if(i == 0) state->pending = 0u;
    if(i >= kMlpParams) return;
    const float gg = g[i];
    g[i] = 0.0f;
    AdamWeight(u, i, gg, a);
}

// ---- weight gradients -------------------------------------------------------
// One block per 16 x 16 tile of dW[k][n] = sum_s X[s][k] dZ[s][n]: its 16 waves
// take every 16th sample tile (one v_mfma_f32_16x16x32_bf16 each; with samples
// contiguous both operands are 1 KiB contiguous loads) and are summed through
// LDS in wave order, so there are no atomics and the sum is deterministic.
// ADAM: the block also updates its 256 parameters, pending gradients included.
// Bound by L2 reads (each operand tile is read by four blocks): 17 us a batch of
// 16384 (17.9 with atomics and LDS transposes, plus the MLP's Adam pass, 4.9).
constexpr uint32_t kWgradWaves = 16;
constexpr uint32_t kWgradBlocks = 8u * 16u;   // an XCD per layer, two of them idle
typedef float v4f __attribute__((ext_vector_type(4)));
template<bool ADAM>
__global__ void __launch_bounds__(kWgradWaves * 64)
KNrcWgrad(NrcTrainBuf tb, uint32_t batch, float* __restrict__ wgrad, MlpAdam u, AdamArgs a)
{
    __shared__ float part[kWgradWaves][256];
    // workgroups go round-robin over the 8 XCDs: a layer's 16 tiles share an L2
    const uint32_t l = blockIdx.x & 7u, kt = blockIdx.x >> 5, nt = (blockIdx.x >> 3) & 3u;
    if(l >= kNrcLayers) return;
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6, tiles = batch / 32u;
    v4f acc = v4f{0};
    const bool apply = ADAM && tb.state->apply != 0u;
    // outputs past the third have no gradient (and none is stored)
    const bool live = l + 1u < kNrcLayers || nt == 0u;
    if(live)
    {
        // lane (r, q): row r of the tile, samples 8 q .. 8 q + 7
        const uint32_t at = (lane & 15u) * 4u + (lane >> 4);
        const uint4* __restrict__ X = reinterpret_cast<const uint4*>(tb.x) + size_t(l) * tiles * 256u + kt * 64u + at;
        const uint4* __restrict__ G = reinterpret_cast<const uint4*>(tb.dz) + size_t(l) * tiles * 256u + nt * 64u + at;
        constexpr uint32_t kAhead = 8;       // tiles whose loads are in flight together
        for(uint32_t t = wave; t < tiles; t += kAhead * kWgradWaves)
        {
            uint4 xv[kAhead], gv[kAhead];
            #pragma unroll
            for(uint32_t j = 0; j < kAhead; j++)
            {
                // past the last tile: that one again, as zeros
                const uint32_t tj = t + j * kWgradWaves, tr = min(tj, tiles - 1u);
                xv[j] = X[size_t(tr) * 256u];
                gv[j] = G[size_t(tr) * 256u];
                if(tj != tr) xv[j] = gv[j] = make_uint4(0u, 0u, 0u, 0u);
            }
            #pragma unroll
            for(uint32_t j = 0; j < kAhead; j++)
                acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8bf, xv[j]),
                                                              __builtin_bit_cast(v8bf, gv[j]), acc, 0, 0, 0);
        }
    }
    // lane (c, q) holds column c, rows 4 q .. 4 q + 3
    for(uint32_t e = 0; e < 4; e++) part[wave][(4u * (lane >> 4) + e) * 16u + (lane & 15u)] = acc[e];
    __syncthreads();
    if(threadIdx.x >= 256u) return;
    float g = 0.0f;
    for(uint32_t w = 0; w < kWgradWaves; w++) g += part[w][threadIdx.x];
    const uint32_t k = kt * 16u + (threadIdx.x >> 4), n = nt * 16u + (threadIdx.x & 15u);
    const uint32_t i = l * kLayerParams + k * kW + n;
    if constexpr(ADAM)
    {
        if(apply) { g += wgrad[i]; wgrad[i] = 0.0f; }
        AdamWeight(u, i, g, a);
    }
    else if(live && g != 0.0f) wgrad[i] += g;
}

// Grid parameters, four at a time (two table entries).  LAZY: entries with a
// zero gradient keep parameter and moments, and are not written.
struct GridAdam
{
    float* p;
    float* m;
    float* v;
    __half* h;
};
template<bool LAZY>
__device__ __forceinline__ void AdamGrid4(const GridAdam& u, size_t i, float4 g4, const AdamArgs& a)
{
    if(LAZY && g4.x == 0.0f && g4.y == 0.0f && g4.z == 0.0f && g4.w == 0.0f) return;
    float4 p4 = reinterpret_cast<const float4*>(u.p)[i];
    float4 m4 = reinterpret_cast<const float4*>(u.m)[i];
    float4 v4 = reinterpret_cast<const float4*>(u.v)[i];
    float* pp = &p4.x;
    float* mm = &m4.x;
    float* v2 = &v4.x;
    float* gg = &g4.x;
    #pragma unroll
    for(int k = 0; k < 4; k++)
        if(!LAZY || gg[k] != 0.0f) AdamOne(pp[k], mm[k], v2[k], gg[k], a);
    reinterpret_cast<float4*>(u.p)[i] = p4;
    reinterpret_cast<float4*>(u.m)[i] = m4;
    reinterpret_cast<float4*>(u.v)[i] = v4;
    reinterpret_cast<__half2*>(u.h)[2 * i] = __floats2half2_rn(p4.x, p4.y);
    reinterpret_cast<__half2*>(u.h)[2 * i + 1] = __floats2half2_rn(p4.z, p4.w);
}

template<bool LAZY>
__global__ void __launch_bounds__(256)
KNrcAdamGrid(GridAdam u, float* __restrict__ g, size_t count, AdamArgs a)
{
    const size_t n4 = count / 4u;
    size_t i = size_t(blockIdx.x) * blockDim.x + threadIdx.x;
    for(; i < n4; i += size_t(gridDim.x) * blockDim.x)
    {
        const float4 g4 = reinterpret_cast<const float4*>(g)[i];
        if(LAZY && g4.x == 0.0f && g4.y == 0.0f && g4.z == 0.0f && g4.w == 0.0f) continue;
        reinterpret_cast<float4*>(g)[i] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        AdamGrid4<LAZY>(u, i, g4, a);
    }
}

// Grid gradient by segments: a block owns kSegEntries entries of one level in
// LDS, scans every sample of the batch for corners that fall inside (an index
// costs a few integer operations, a global float atomic into a table that no
// L2 holds about 0.05 ns of the whole chip), adds them with LDS atomics and
// then either adds the segment to the gradient buffer or, in a training step,
// runs Adam on it, so that the gradient never goes to memory.
// 8192 entries: 64 KiB of LDS, two workgroups per CU; a level has at least 32
// segments, because a small level's corners all fall into its few entries.
// 16384 samples, 16 levels of 2^19: 83 us with Adam (its parameters and
// moments, 26 B each, take 61 us at the card's copy rate), from 245 us of
// atomics and 97 us of Adam; with one segment for each small level 336 us.
constexpr uint32_t kSegEntries = 8192;
constexpr uint32_t kSegMinPerLevel = 32;
constexpr uint32_t kOwnerTPB = 1024;
// Segments of one level up to which the scan is the faster way: it costs
// every sample about 4 ps a segment, the 16 atomics about 0.8 ns.
constexpr uint32_t kOwnerMaxSegs = 128;
struct OwnerLevels
{
    uint32_t first[kNrcMaxLevels + 1];   // first block of each level
    uint32_t used[kNrcMaxLevels];        // entries an index can reach
    uint32_t size[kNrcMaxLevels];        // entries of a segment (even)
};
enum : int { OWNER_ADD = 0, OWNER_ADAM = 1, OWNER_LAZY = 2 };
template<int MODE>
__global__ void __launch_bounds__(kOwnerTPB)
KNrcGridOwner(NrcView v, NrcTrainBuf tb, uint32_t batch, OwnerLevels ol, float* __restrict__ ggrad,
              GridAdam u, AdamArgs a)
{
    __shared__ __attribute__((aligned(16))) float seg[kSegEntries * 2u];
    uint32_t l = 0;
    while(blockIdx.x >= ol.first[l + 1]) l++;
    const uint32_t base = (blockIdx.x - ol.first[l]) * ol.size[l];
    const uint32_t count = min(ol.size[l], ol.used[l] - base);
    const size_t first = ((size_t(l) << v.log2T) + base) / 2u;      // in pairs of entries
    const bool apply = MODE != OWNER_ADD && tb.state->apply != 0u;
    for(uint32_t e = threadIdx.x; e < (count + 1u) / 2u; e += kOwnerTPB)
        reinterpret_cast<float4*>(seg)[e] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    __syncthreads();
    const uint32_t mask = (1u << v.log2T) - 1u, dense = v.dense[l], dy = v.my[l], dz = v.mz[l];
    const float scale = v.scale[l];
    for(uint32_t s = threadIdx.x; s < batch; s += kOwnerTPB)
    {
        const float2 g = tb.dx0[size_t(l) * batch + s];
        const float pos[3] = {tb.pos[s], tb.pos[batch + s], tb.pos[2 * size_t(batch) + s]};
        const Cell c = LevelCell(pos, scale, dy, dz);
        // the two corners along x differ in the low index bits only, so a
        // pair mostly falls in or out together
        #pragma unroll
        for(uint32_t q = 0; q < 4; q++)
        {
            const uint32_t y = c.y + ((q & 1u) ? dy : 0u), z = c.z + ((q & 2u) ? dz : 0u);
            const uint32_t i0 = GridIndex(dense, mask, c.x, y, z) - base;
            const uint32_t i1 = GridIndex(dense, mask, c.x + 1u, y, z) - base;
            if(min(i0, i1) >= count) continue;
            const float w0 = CornerWeight(c, 2u * q), w1 = CornerWeight(c, 2u * q + 1u);
            if(i0 < count)
            {
                atomicAdd(&seg[2u * i0], w0 * g.x);
                atomicAdd(&seg[2u * i0 + 1u], w0 * g.y);
            }
            if(i1 < count)
            {
                atomicAdd(&seg[2u * i1], w1 * g.x);
                atomicAdd(&seg[2u * i1 + 1u], w1 * g.y);
            }
        }
    }
    __syncthreads();
    for(uint32_t e = threadIdx.x; e < (count + 1u) / 2u; e += kOwnerTPB)
    {
        float4 g4 = reinterpret_cast<const float4*>(seg)[e];
        if constexpr(MODE == OWNER_ADD)
        {
            if(g4.x == 0.0f && g4.y == 0.0f && g4.z == 0.0f && g4.w == 0.0f) continue;
            float4 t = reinterpret_cast<const float4*>(ggrad)[first + e];
            t.x += g4.x; t.y += g4.y; t.z += g4.z; t.w += g4.w;
            reinterpret_cast<float4*>(ggrad)[first + e] = t;
        }
        else
        {
            if(apply)
            {
                const float4 t = reinterpret_cast<const float4*>(ggrad)[first + e];
                g4.x += t.x; g4.y += t.y; g4.z += t.z; g4.w += t.w;
                reinterpret_cast<float4*>(ggrad)[first + e] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            }
            AdamGrid4<MODE == OWNER_LAZY>(u, first + e, g4, a);
        }
    }
}

__global__ void KNrcZero(float* __restrict__ p, size_t n)
{
    size_t i = size_t(blockIdx.x) * blockDim.x + threadIdx.x;
    for(; i < n; i += size_t(gridDim.x) * blockDim.x) p[i] = 0.0f;
}

__global__ void KNrcRefresh(const float* __restrict__ w, uint16_t* __restrict__ wT,
                            uint16_t* __restrict__ wK, const float* __restrict__ grid,
                            __half* __restrict__ h, size_t gridCount)
{
    size_t i = size_t(blockIdx.x) * blockDim.x + threadIdx.x;
    for(size_t j = i; j < kMlpParams; j += size_t(gridDim.x) * blockDim.x)
    {
        uint32_t l = uint32_t(j / kLayerParams), e = uint32_t(j % kLayerParams);
        uint32_t k = e / kW, n = e % kW;
        StoreWeight(wT, wK, l, k, n, w[j]);
    }
    for(size_t j = i; j < gridCount; j += size_t(gridDim.x) * blockDim.x) h[j] = __float2half(grid[j]);
}

} // namespace mray

// ===========================================================================
// Object + C-ABI
// ===========================================================================
using namespace mray;

// Features of one chunk of queries (InferSplit), between the encoding and the
// layers of one call.  All caches of a GPU share its areas (an area in each, 32
// MiB, is never used by a renderer's caches, whose counts only the device knows:
// 1 GiB for 32 views), and calls on up to kFeatAreas streams have one each, so
// that they overlap.  Released with the GPU's last cache.
// 16 levels of 2^19 entries, one call on each of 4 streams: 256 queries 84-100 us
// with one area, 30 with four; 4096 96 -> 42; 16384 113 -> 44; 65536 179 -> 129;
// 131072 265 -> 241.
constexpr uint32_t kFeatAreas = 4;
// Larger calls fill the GPU by themselves and take turns in the first area: side
// by side they share the L2s that the encoding counts on.  On 4 streams, taking
// turns against side by side: 196608 queries 344 / 364 us, 262144 429 / 451,
// 10^6 1428 / 1500 (on two streams 711 / 773).
constexpr uint32_t kOverlapMax = 1u << 17;
// Queries up to which the one-kernel form is taken: its one launch costs the
// host less than two launches, a wait and an event.  64 queries 11.3 us on one
// stream against 11.8, on four 17.5 against 42; 128 on one stream 12.5 against 11.7.
constexpr uint32_t kOneKernelMax = 64;
// The same while several streams query: 256 on two 19.5 us against 19.3, on
// four 18.9 against 40 (on one 14.7 against 12.3); 512 on two 27 against 19.
constexpr uint32_t kOneKernelMaxStreams = 256;
struct FeatArea
{
    uint32_t* feat = nullptr;
    hipEvent_t done = nullptr;    // the area's last use
    hipStream_t stream = nullptr; // of that use: a hint only, calls wait for the event
    uint64_t used = 0;            // its number among the GPU's uses, 0: none yet
};
struct FeatPool
{
    uint32_t caches = 0;
    uint64_t uses = 0;
    FeatArea area[kFeatAreas];
};
// Never destroyed: a program's own static objects may end their caches late.
static std::mutex& featLock = *new std::mutex();             // every pool
static std::map<int, FeatPool>& featPools = *new std::map<int, FeatPool>();

static bool AllocFeatArea(FeatArea& a)
{
    if(a.feat) return true;
    // no stream operation: another thread's capture is none of its concern
    hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
    (void)hipThreadExchangeStreamCaptureMode(&mode);
    void* p = nullptr;
    if(hipMalloc(&p, size_t(kSplitChunk) * kNrcMaxLevels * 4u) == hipSuccess)
    {
        if(hipEventCreateWithFlags(&a.done, hipEventDisableTiming) == hipSuccess) a.feat = static_cast<uint32_t*>(p);
        else (void)hipFree(p);
    }
    (void)hipThreadExchangeStreamCaptureMode(&mode);
    if(!a.feat) (void)hipGetLastError();
    return a.feat != nullptr;
}

static void ReleaseFeatPool(int device)
{
    std::lock_guard<std::mutex> lock(featLock);
    FeatPool& p = featPools[device];
    if(--p.caches != 0u) return;
    for(FeatArea& a : p.area)
    {
        if(!a.feat) continue;
        (void)hipEventSynchronize(a.done);
        (void)hipEventDestroy(a.done);
        (void)hipFree(a.feat);
    }
    featPools.erase(device);
}

struct MRayNrc
{
    MRayNrcConfig cfg{};
    int device = -1;              // whose pool it uses
    DeviceArena arena;
    NrcView view{};
    uint16_t* wT = nullptr;
    uint16_t* wK = nullptr;
    float* w = nullptr;
    float* wm = nullptr;
    float* wv = nullptr;
    float* wg = nullptr;
    __half* gridH = nullptr;
    float* grid = nullptr;
    float* gm = nullptr;
    float* gv = nullptr;
    float* gg = nullptr;
    size_t gridCount = 0;
    NrcTrainBuf tb{};
    uint32_t maxBatch = 0;
    uint64_t step = 0;
    uint32_t inferBlocks = 0;     // resident inference blocks
    OwnerLevels owner{};
    uint32_t ownerSegs = 0;       // segments of the largest level
    EncodePlan plan{};
    // per-kernel timing (mray_nrc_set_profiling): event pairs around each
    // launch, harvested by mray_nrc_kernel_times
    bool profiling = false;
    std::vector<hipEvent_t> evPool;
    std::vector<std::pair<uint32_t, std::pair<hipEvent_t, hipEvent_t>>> evPending;
    double kMs[kNrcKernelKinds] = {};
    uint64_t kLaunches[kNrcKernelKinds] = {};
};

// Event pair around one launch of kernel kind k (profiling only).
struct NrcTimer
{
    MRayNrc* n;
    uint32_t k;
    hipStream_t s;
    hipEvent_t a = nullptr, b = nullptr;
    NrcTimer(MRayNrc* n_, uint32_t k_, hipStream_t s_) : n(n_), k(k_), s(s_)
    {
        if(!n->profiling) return;
        a = Take();
        b = Take();
        if(a && b) (void)hipEventRecord(a, s);
    }
    ~NrcTimer()
    {
        if(!a || !b) return;
        (void)hipEventRecord(b, s);
        n->evPending.push_back({k, {a, b}});
    }
    hipEvent_t Take()
    {
        if(!n->evPool.empty()) { hipEvent_t e = n->evPool.back(); n->evPool.pop_back(); return e; }
        hipEvent_t e = nullptr;
        return (hipEventCreate(&e) == hipSuccess) ? e : nullptr;
    }
};

static int NrcLaunchCheck() { MRAY_HIP_CHECK(hipGetLastError()); return MRAY_OK; }


extern "C" {

int mray_nrc_create(const MRayNrcConfig* hCfg, MRayNrc** out)
{
    if(!hCfg || !out) { SetError("nrc_create: NULL argument"); return MRAY_ERR_INVALID; }
    *out = nullptr;
    const MRayNrcConfig& c = *hCfg;
    if(c.levels == 0 || c.levels > kNrcMaxLevels || c.log2TableSize < 10 || c.log2TableSize > 24 ||
       c.minResolution < 2 || c.maxResolution < c.minResolution || c.maxBatch == 0 ||
       (c.maxBatch % 32u) != 0)
    {
        SetError("nrc_create: levels 1..16, log2TableSize 10..24, 2 <= minRes <= maxRes, "
                 "maxBatch a non-zero multiple of 32");
        return MRAY_ERR_INVALID;
    }
    MRayNrc* n = new MRayNrc();
    n->cfg = c;
    NrcView& v = n->view;
    v.levels = c.levels;
    v.log2T = c.log2TableSize;
    const double b = (c.levels > 1)
        ? std::exp((std::log(double(c.maxResolution)) - std::log(double(c.minResolution))) / (c.levels - 1))
        : 1.0;
    for(uint32_t l = 0; l < kNrcMaxLevels; l++)
    {
        float s = (l < c.levels) ? float(double(c.minResolution) * std::pow(b, double(l)) - 1.0) : 1.0f;
        v.scale[l] = s;
        const uint32_t res = uint32_t(std::ceil(s)) + 2u;
        const uint64_t cells = uint64_t(res) * res * res;
        v.dense[l] = (cells <= (1ull << c.log2TableSize)) ? 1u : 0u;
        v.my[l] = v.dense[l] ? res : 2654435761u;
        v.mz[l] = v.dense[l] ? res * res : 805459861u;
        // entries an index of this level reaches.  The rest of a dense level's
        // table never gets a gradient, and Adam on zero moments leaves it as
        // it is (with eps = 0 it would not: 0 / 0)
        const uint64_t used = (v.dense[l] && c.epsilon > 0.0f) ? cells : (1ull << c.log2TableSize);
        n->owner.used[l] = uint32_t(used);
        const uint32_t size = std::min(kSegEntries, (DivUp(used, kSegMinPerLevel) + 1u) & ~1u);
        n->owner.size[l] = size;
        const uint32_t segs = (l < c.levels) ? DivUp(used, size) : 0u;
        n->owner.first[l + 1] = n->owner.first[l] + segs;
        n->ownerSegs = std::max(n->ownerSegs, segs);
    }
    // encoding plan: whole rows of 8 hashed levels, one per XCD; the rest shared
    {
        std::vector<uint32_t> hashed, rest;
        for(uint32_t l = 0; l < c.levels; l++) (v.dense[l] ? rest : hashed).push_back(l);
        EncodePlan& p = n->plan;
        p.own = uint32_t(hashed.size()) / 8u;
        for(uint32_t k = 0; k < 8u * p.own; k++) p.ownLevel[k] = hashed[hashed.size() - 1u - k];
        for(size_t k = 0; k + 8u * p.own < hashed.size(); k++) rest.push_back(hashed[k]);
        p.shared = uint32_t(rest.size());
        std::copy(rest.begin(), rest.end(), p.sharedLevel);
    }
    n->gridCount = size_t(c.levels) << c.log2TableSize;
    n->gridCount *= kNrcFeat;
    n->maxBatch = c.maxBatch;
    auto A = [&](void** p, size_t bytes) { return DevAlloc(n->arena, p, bytes); };
    int rv = MRAY_OK;
    auto fail = [&](int r) { n->arena.Release(); if(n->device >= 0) ReleaseFeatPool(n->device); delete n; return r; };
    int dev = 0;
    if(hipGetDevice(&dev) != hipSuccess) return fail(MRAY_ERR_HIP);
    {
        // the first area now, not in some call's first pass; without memory
        // for it queries take the one-kernel form
        std::lock_guard<std::mutex> lock(featLock);
        FeatPool& p = featPools[dev];
        p.caches++;
        n->device = dev;
        (void)AllocFeatArea(p.area[0]);
    }
    if((rv = A((void**)&n->wT, kMlpParams * 2)) != MRAY_OK) return fail(rv);
    if((rv = A((void**)&n->wK, kMlpParams * 2)) != MRAY_OK) return fail(rv);
    if((rv = A((void**)&n->w, kMlpParams * 4)) != MRAY_OK) return fail(rv);
    if((rv = A((void**)&n->wm, kMlpParams * 4)) != MRAY_OK) return fail(rv);
    if((rv = A((void**)&n->wv, kMlpParams * 4)) != MRAY_OK) return fail(rv);
    if((rv = A((void**)&n->wg, kMlpParams * 4)) != MRAY_OK) return fail(rv);
    if((rv = A((void**)&n->gridH, n->gridCount * 2)) != MRAY_OK) return fail(rv);
    if((rv = A((void**)&n->grid, n->gridCount * 4)) != MRAY_OK) return fail(rv);
    if((rv = A((void**)&n->gm, n->gridCount * 4)) != MRAY_OK) return fail(rv);
    if((rv = A((void**)&n->gv, n->gridCount * 4)) != MRAY_OK) return fail(rv);
    if((rv = A((void**)&n->gg, n->gridCount * 4)) != MRAY_OK) return fail(rv);
    const size_t B = c.maxBatch;
    if((rv = A((void**)&n->tb.x, kNrcLayers * B * kW * 2)) != MRAY_OK) return fail(rv);
    if((rv = A((void**)&n->tb.dz, kNrcLayers * B * kW * 2)) != MRAY_OK) return fail(rv);
    if((rv = A((void**)&n->tb.dx0, B * 32 * 4)) != MRAY_OK) return fail(rv);
    if((rv = A((void**)&n->tb.pos, B * 3 * 4)) != MRAY_OK) return fail(rv);
    if((rv = A((void**)&n->tb.loss, B / 32 * 4)) != MRAY_OK) return fail(rv);
    if((rv = A((void**)&n->tb.state, sizeof(NrcState))) != MRAY_OK) return fail(rv);
    v.wT = n->wT;
    v.wK = n->wK;
    v.grid = n->gridH;
    // initial parameters: grid U(-1e-4, 1e-4); layers U(-a, a), a = sqrt(6/(in+out))
    // (Glorot); the output layer keeps only columns 0..2
    {
        std::mt19937 mt(uint32_t(c.seed ^ (c.seed >> 32)));
        std::uniform_real_distribution<float> ug(-1e-4f, 1e-4f);
        std::vector<float> hg(n->gridCount);
        for(float& x : hg) x = ug(mt);
        std::vector<float> hw(kMlpParams, 0.0f);
        for(uint32_t l = 0; l < kNrcLayers; l++)
        {
            uint32_t fanOut = (l + 1 == kNrcLayers) ? 3u : kW;
            float a = std::sqrt(6.0f / float(kW + fanOut));
            std::uniform_real_distribution<float> uw(-a, a);
            for(uint32_t k = 0; k < kW; k++)
                for(uint32_t o = 0; o < fanOut; o++) hw[l * kLayerParams + k * kW + o] = uw(mt);
        }
        if(hipMemcpy(n->grid, hg.data(), n->gridCount * 4, hipMemcpyHostToDevice) != hipSuccess ||
           hipMemcpy(n->w, hw.data(), kMlpParams * 4, hipMemcpyHostToDevice) != hipSuccess)
        {
            SetError("nrc_create: upload failed");
            return fail(MRAY_ERR_HIP);
        }
    }
    KNrcZero<<<256, 256>>>(n->wm, kMlpParams);
    KNrcZero<<<256, 256>>>(n->wv, kMlpParams);
    KNrcZero<<<256, 256>>>(n->wg, kMlpParams);
    KNrcZero<<<1, 64>>>(reinterpret_cast<float*>(n->tb.state), sizeof(NrcState) / 4u);
    KNrcZero<<<2048, 256>>>(n->gm, n->gridCount);
    KNrcZero<<<2048, 256>>>(n->gv, n->gridCount);
    KNrcZero<<<2048, 256>>>(n->gg, n->gridCount);
    KNrcRefresh<<<2048, 256>>>(n->w, n->wT, n->wK, n->grid, n->gridH, n->gridCount);
    if(hipDeviceSynchronize() != hipSuccess || hipGetLastError() != hipSuccess)
    {
        SetError("nrc_create: initialisation kernels failed");
        return fail(MRAY_ERR_HIP);
    }
    hipDeviceProp_t prop;
    if(hipGetDeviceProperties(&prop, dev) != hipSuccess) return fail(MRAY_ERR_HIP);
    int perCu = 0;
    if(hipOccupancyMaxActiveBlocksPerMultiprocessor(&perCu, KNrcInfer, int(kInferTPB), 0) != hipSuccess || perCu < 1)
        perCu = 1;
    n->inferBlocks = uint32_t(std::max(1, prop.multiProcessorCount)) * uint32_t(perCu);
    *out = n;
    return MRAY_OK;
}

int mray_nrc_destroy(MRayNrc* n)
{
    if(!n) return MRAY_OK;
    (void)hipDeviceSynchronize();
    for(auto& p : n->evPending)
    {
        (void)hipEventDestroy(p.second.first);
        (void)hipEventDestroy(p.second.second);
    }
    for(hipEvent_t e : n->evPool) (void)hipEventDestroy(e);
    n->arena.Release();
    ReleaseFeatPool(n->device);
    delete n;
    return MRAY_OK;
}

// Encoding in its own pass, chunk by chunk through an area of the GPU's pool.
// A call takes the area of its stream's last call, else one not used yet, else
// the one whose last use is longest ago (large ones the first, kOverlapMax), and
// waits for that area's last use.  A call under
// capture (its graph may run beside others) takes the one-kernel form, and so
// do small ones (kOneKernelMax) and one that finds no memory for an area.
constexpr int kNoSplit = -1;
static int InferSplit(MRayNrc* n, const float* dRecords, uint32_t count, float* dOut, uint32_t blocks, hipStream_t s)
{
    if(count <= kOneKernelMax) return kNoSplit;
    hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
    MRAY_HIP_CHECK(hipStreamIsCapturing(s, &cap));
    if(cap != hipStreamCaptureStatusNone) return kNoSplit;
    std::lock_guard<std::mutex> lock(featLock);
    FeatPool& pool = featPools[n->device];
    if(count <= kOneKernelMaxStreams && pool.area[1].used != 0u) return kNoSplit;
    FeatArea* a = &pool.area[0];
    for(FeatArea& c : pool.area)
    {
        if(count > kOverlapMax) break;
        if(c.used && c.stream == s) { a = &c; break; }
        if(c.used < a->used) a = &c;
    }
    int dev = n->device;
    if(!a->feat)
    {
        (void)hipGetDevice(&dev);
        if(dev != n->device) (void)hipSetDevice(n->device);
        const bool ok = AllocFeatArea(*a);
        if(dev != n->device) (void)hipSetDevice(dev);
        if(!ok) return kNoSplit;
    }
    a->stream = s;
    a->used = ++pool.uses;
    MRAY_HIP_CHECK(hipStreamWaitEvent(s, a->done, 0));
    const EncodePlan& p = n->plan;
    for(uint32_t at = 0; at < count; at += kSplitChunk)
    {
        const uint32_t c = std::min(kSplitChunk, count - at);
        const uint32_t b = DivUp(c, kEncodeTPB), perXcd = p.own * b + p.shared * DivUp(b, 8u);
        const float* rec = dRecords + size_t(at) * 11u;
        NrcTimer t(n, 0, s);
        KNrcEncode<<<8u * perXcd, kEncodeTPB, 0, s>>>(n->view, rec, c, p, a->feat);
        KNrcInferEncoded<<<blocks, kInferTPB, 0, s>>>(n->view, rec, a->feat, c, dOut + size_t(at) * 3u);
    }
    MRAY_HIP_CHECK(hipEventRecord(a->done, s));
    return NrcLaunchCheck();
}

int mray_nrc_infer(MRayNrc* n, const float* dRecords, uint32_t count, const uint32_t* dCount,
                   float* dOut, void* stream)
{
    if(!n || !dRecords || !dOut) { SetError("nrc_infer: NULL argument"); return MRAY_ERR_INVALID; }
    hipStream_t s = static_cast<hipStream_t>(stream);
    const uint32_t all = DivUp(std::max(count, 1u), 32u * (kInferTPB / 64u));
    const uint32_t blocks = dCount ? n->inferBlocks : std::min(n->inferBlocks, all);
    if(!dCount && count > 0)
    {
        const int r = InferSplit(n, dRecords, count, dOut, blocks, s);
        if(r != kNoSplit) return r;
    }
    {
        NrcTimer t(n, 0, s);
        KNrcInfer<<<blocks, kInferTPB, 0, s>>>(n->view, dRecords, dCount, count, dOut);
    }
    return NrcLaunchCheck();
}

static MlpAdam MlpOf(const MRayNrc* n) { return {n->w, n->wm, n->wv, n->wT, n->wK}; }
static GridAdam GridOf(const MRayNrc* n) { return {n->grid, n->gm, n->gv, n->gridH}; }

static AdamArgs NextAdam(MRayNrc* n)
{
    n->step++;
    AdamArgs a;
    a.lr = n->cfg.learningRate;
    a.b1 = n->cfg.beta1;
    a.b2 = n->cfg.beta2;
    a.eps = n->cfg.epsilon;
    a.c1 = float(1.0 / (1.0 - std::pow(double(a.b1), double(n->step))));
    a.c2 = float(1.0 / (1.0 - std::pow(double(a.b2), double(n->step))));
    return a;
}

static int CheckBatch(const MRayNrc* n, const float* dRecords, const float* dTargets, uint32_t count)
{
    if(!n || !dRecords || !dTargets) { SetError("nrc_backward: NULL argument"); return MRAY_ERR_INVALID; }
    if(count == 0 || count > n->maxBatch || (count % 32u) != 0)
    {
        SetError("nrc_backward: count must be a non-zero multiple of 32, at most maxBatch");
        return MRAY_ERR_INVALID;
    }
    return MRAY_OK;
}

// Forward and data gradients of one batch.
static void LaunchTrain(MRayNrc* n, const float* dRecords, const float* dTargets, uint32_t count, uint32_t step,
                        hipStream_t s)
{
    NrcTimer t(n, 1, s);
    KNrcTrain<<<count / 32u, 64, 0, s>>>(n->view, dRecords, dTargets, n->tb, count, step);
}

int mray_nrc_backward(MRayNrc* n, const float* dRecords, const float* dTargets, uint32_t count,
                      void* stream)
{
    MRAY_TRY(CheckBatch(n, dRecords, dTargets, count));
    hipStream_t s = static_cast<hipStream_t>(stream);
    LaunchTrain(n, dRecords, dTargets, count, 0u, s);
    {
        NrcTimer t(n, 3, s);
        KNrcWgrad<false><<<kWgradBlocks, kWgradWaves * 64, 0, s>>>(n->tb, count, n->wg, MlpAdam{}, AdamArgs{});
    }
    {
        NrcTimer t(n, 4, s);
        // the segments' fixed cost (clearing and reading all of them, about
        // 10 us) is that of the atomics of about 1000 samples
        if(n->ownerSegs <= kOwnerMaxSegs && count >= 1024u)
            KNrcGridOwner<OWNER_ADD><<<n->owner.first[kNrcMaxLevels], kOwnerTPB, 0, s>>>(
                n->view, n->tb, count, n->owner, n->gg, GridAdam{}, AdamArgs{});
        else
            KNrcGridBwd<<<dim3(DivUp(count, 256u), n->view.levels), 256, 0, s>>>(n->view, n->tb, count, n->gg);
    }
    return NrcLaunchCheck();
}

int mray_nrc_adam(MRayNrc* n, void* stream)
{
    if(!n) { SetError("nrc_adam: NULL argument"); return MRAY_ERR_INVALID; }
    hipStream_t s = static_cast<hipStream_t>(stream);
    const AdamArgs a = NextAdam(n);
    NrcTimer t(n, 5, s);
    KNrcAdamMlp<<<DivUp(kMlpParams, 256u), 256, 0, s>>>(MlpOf(n), n->wg, a, n->tb.state);
    if(n->cfg.flags & MRAY_NRC_LAZY_ADAM)
        KNrcAdamGrid<true><<<4096, 256, 0, s>>>(GridOf(n), n->gg, n->gridCount, a);
    else
        KNrcAdamGrid<false><<<4096, 256, 0, s>>>(GridOf(n), n->gg, n->gridCount, a);
    return NrcLaunchCheck();
}

// Backward and Adam.  Both gradients are applied where they are formed and
// never stored, together with what earlier backward passes left pending.
int mray_nrc_train(MRayNrc* n, const float* dRecords, const float* dTargets, uint32_t count,
                   void* stream)
{
    MRAY_TRY(CheckBatch(n, dRecords, dTargets, count));
    if(n->ownerSegs > kOwnerMaxSegs)
    {
        MRAY_TRY(mray_nrc_backward(n, dRecords, dTargets, count, stream));
        return mray_nrc_adam(n, stream);
    }
    hipStream_t s = static_cast<hipStream_t>(stream);
    LaunchTrain(n, dRecords, dTargets, count, 1u, s);
    const AdamArgs a = NextAdam(n);
    {
        NrcTimer t(n, 3, s);
        KNrcWgrad<true><<<kWgradBlocks, kWgradWaves * 64, 0, s>>>(n->tb, count, n->wg, MlpOf(n), a);
    }
    {
        NrcTimer t(n, 4, s);
        const uint32_t blocks = n->owner.first[kNrcMaxLevels];
        if(n->cfg.flags & MRAY_NRC_LAZY_ADAM)
            KNrcGridOwner<OWNER_LAZY><<<blocks, kOwnerTPB, 0, s>>>(n->view, n->tb, count, n->owner, n->gg, GridOf(n), a);
        else
            KNrcGridOwner<OWNER_ADAM><<<blocks, kOwnerTPB, 0, s>>>(n->view, n->tb, count, n->owner, n->gg, GridOf(n), a);
    }
    return NrcLaunchCheck();
}

int mray_nrc_last_loss(MRayNrc* n, float* hLoss)
{
    if(!n || !hLoss) { SetError("nrc_last_loss: NULL argument"); return MRAY_ERR_INVALID; }
    MRAY_HIP_CHECK(hipDeviceSynchronize());
    NrcState state{};
    MRAY_HIP_CHECK(hipMemcpy(&state, n->tb.state, sizeof(state), hipMemcpyDeviceToHost));
    std::vector<float> part(state.tiles);
    MRAY_HIP_CHECK(hipMemcpy(part.data(), n->tb.loss, part.size() * sizeof(float), hipMemcpyDeviceToHost));
    double sum = 0.0;
    for(float x : part) sum += x;
    *hLoss = float(sum);
    return MRAY_OK;
}

int mray_nrc_param_counts(const MRayNrc* n, uint64_t* hMlp, uint64_t* hGrid)
{
    if(!n || !hMlp || !hGrid) { SetError("nrc_param_counts: NULL argument"); return MRAY_ERR_INVALID; }
    *hMlp = kMlpParams;
    *hGrid = n->gridCount;
    return MRAY_OK;
}

int mray_nrc_read(MRayNrc* n, uint32_t which, float* hOut)
{
    if(!n || !hOut) { SetError("nrc_read: NULL argument"); return MRAY_ERR_INVALID; }
    MRAY_HIP_CHECK(hipDeviceSynchronize());
    const float* src = nullptr;
    size_t cnt = 0;
    switch(which)
    {
        case MRAY_NRC_WEIGHTS: src = n->w; cnt = kMlpParams; break;
        case MRAY_NRC_WEIGHT_GRADS: src = n->wg; cnt = kMlpParams; break;
        case MRAY_NRC_GRID: src = n->grid; cnt = n->gridCount; break;
        case MRAY_NRC_GRID_GRADS: src = n->gg; cnt = n->gridCount; break;
        default: SetError("nrc_read: unknown buffer"); return MRAY_ERR_INVALID;
    }
    MRAY_HIP_CHECK(hipMemcpy(hOut, src, cnt * 4, hipMemcpyDeviceToHost));
    return MRAY_OK;
}

int mray_nrc_write(MRayNrc* n, uint32_t which, const float* hIn)
{
    if(!n || !hIn) { SetError("nrc_write: NULL argument"); return MRAY_ERR_INVALID; }
    MRAY_HIP_CHECK(hipDeviceSynchronize());
    if(which == MRAY_NRC_WEIGHTS)
        MRAY_HIP_CHECK(hipMemcpy(n->w, hIn, kMlpParams * 4, hipMemcpyHostToDevice));
    else if(which == MRAY_NRC_GRID)
        MRAY_HIP_CHECK(hipMemcpy(n->grid, hIn, n->gridCount * 4, hipMemcpyHostToDevice));
    else { SetError("nrc_write: only weights and grid are writable"); return MRAY_ERR_INVALID; }
    KNrcRefresh<<<2048, 256>>>(n->w, n->wT, n->wK, n->grid, n->gridH, n->gridCount);
    MRAY_HIP_CHECK(hipGetLastError());
    MRAY_HIP_CHECK(hipDeviceSynchronize());
    return MRAY_OK;
}

int mray_nrc_set_profiling(MRayNrc* n, uint32_t on)
{
    if(!n) { SetError("nrc_set_profiling: NULL argument"); return MRAY_ERR_INVALID; }
    n->profiling = on != 0;
    return MRAY_OK;
}

int mray_nrc_kernel_times(MRayNrc* n, double* hMs, uint64_t* hLaunches)
{
    if(!n || !hMs || !hLaunches) { SetError("nrc_kernel_times: NULL argument"); return MRAY_ERR_INVALID; }
    MRAY_HIP_CHECK(hipDeviceSynchronize());
    for(auto& p : n->evPending)
    {
        float ms = 0.0f;
        MRAY_HIP_CHECK(hipEventElapsedTime(&ms, p.second.first, p.second.second));
        n->kMs[p.first] += ms;
        n->kLaunches[p.first] += 1;
        n->evPool.push_back(p.second.first);
        n->evPool.push_back(p.second.second);
    }
    n->evPending.clear();
    for(uint32_t k = 0; k < kNrcKernelKinds; k++)
    {
        hMs[k] = n->kMs[k];
        hLaunches[k] = n->kLaunches[k];
    }
    return MRAY_OK;
}

int mray_nrc_zero_grads(MRayNrc* n, void* stream)
{
    if(!n) { SetError("nrc_zero_grads: NULL argument"); return MRAY_ERR_INVALID; }
    hipStream_t s = static_cast<hipStream_t>(stream);
    KNrcZero<<<256, 256, 0, s>>>(n->wg, kMlpParams);
    KNrcZero<<<2048, 256, 0, s>>>(n->gg, n->gridCount);
    KNrcZero<<<1, 64, 0, s>>>(reinterpret_cast<float*>(&n->tb.state->pending), 1u);
    return NrcLaunchCheck();
}

} // extern "C"
