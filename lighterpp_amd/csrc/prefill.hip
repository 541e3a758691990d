// prefill.hip -- batched prefill: the key/value cache entries of a run of prompt
// tokens in one pass over the weights.
//
// The reference has no such path: it prefills by decoding the prompt one token at
// a time and dropping what the sampler returns (src/main.cpp:163-180), which reads
// every weight once per prompt token.  Here the prompt's tokens go through each
// layer together, so the matrix products are GEMMs on the matrix cores
// (v_mfma_f32_16x16x32_f16 and 32x32x16) and every weight is read once per chunk of up to 2048
// tokens.  What a prefill leaves behind is exactly what the decode loop reads
// later: K and V of the prompt positions, rounded to binary16 as the cache store
// rounds them (model.cpp:171-176, kernels.cuh:34).  The classifier and the sampler
// are not run: the ids they would produce are the ones main.cpp drops.
//
// Arithmetic: weights binary16 as stored; activations fp32, split for the matrix
// cores into a binary16 head and a binary16 remainder (x = hi + lo to about 2^-22),
// both multiplied into the same fp32 accumulators; everything between the GEMMs
// (RMSNorm, RoPE, softmax, SwiGLU, residual) in fp32 with the operators' own
// operation order (ops.cpp:20-87).
#include <cmath>
#include <cstdlib>
#include <type_traits>

#include "lpp_device.hpp"
#include "lpp_internal.hpp"
#include "lpp_model.hpp"

namespace lpp {
namespace pf {

using namespace dev;

typedef float floatx16 __attribute__((ext_vector_type(16)));

constexpr int kTileTokens = 128;    // token rows of a workgroup's output tile
constexpr int kTileFeatures = 128;  // weight rows of it
// Prompt tokens per pass over the weights, at most.  What a longer chunk saves is the ends of launches: 512 tokens give the
// 1B shape's W1+W3 one tile per compute unit, whose first data and epilogue (12 of 69 us) overlap nothing, and its other
// products less than that; norm, RoPE and attention are then launches of 5 to 15 us.  1B shape, exact mode, chunks of at
// most 512 / 1024 / 2048 / 3072: 2011 ids 10.9 / 9.1 / 8.5 / 8.5 ms, 6000 ids 37.7 / 30.4 / 28.5 / 29.9; fast mode, 2011
// ids: 8.4 / 6.6 / 5.9 / 5.9.  8B shape, 2011 ids: 60.6 / 57.3 / 53.6 ms.
constexpr int kChunk = 2048;
constexpr int kSmallChunk = 512;  // where device memory has no room for the buffers of more
constexpr int kMaxGqa = 8;          // query heads per KV head the attention kernel keeps in registers

// ---------------------------------------------------------------------------
// Small per-token kernels
// ---------------------------------------------------------------------------

// x[t][:] = embedding row of tokens[t] (model.cpp:346-348).
__global__ __launch_bounds__(256) void k_embed(const float* __restrict__ emb, const int* __restrict__ tokens,
                                               float* __restrict__ x, int dim) {
    const int t = blockIdx.x;
    const float* src = emb + static_cast<size_t>(tokens[t]) * dim;
    for (int i = threadIdx.x; i < dim; i += blockDim.x) x[static_cast<size_t>(t) * dim + i] = src[i];
}

__device__ __forceinline__ float block_sum256(float v, float* scratch) {
    v = wave_sum(v);
    if (lane_id() == 0) scratch[threadIdx.x / kWave] = v;
    __syncthreads();
    const float total = (scratch[0] + scratch[1]) + (scratch[2] + scratch[3]);
    __syncthreads();
    return total;
}

__device__ __forceinline__ void split_store(half_t* hi, half_t* lo, size_t at, float v) {
    const half_t h = static_cast<half_t>(v);
    hi[at] = h;
    lo[at] = static_cast<half_t>(v - static_cast<float>(h));
}

// (hi, lo)[t][:] = RMSNorm(x[t][:]) * gain (ops.cpp:20-32); rows t >= n_tokens are zero.
// With `splits` > 0 the residual update that precedes the norm is done here: x[t][:] += p[0][t][:] +
// p[1][t][:] + ... in that order, the partial products of a GEMM whose K was split (p[z] starts at
// partials + z * split_stride), written back to x.
__global__ __launch_bounds__(256) void k_norm_split(float* __restrict__ x, const float* __restrict__ gain,
                                                    half_t* __restrict__ hi, half_t* __restrict__ lo, int dim,
                                                    int n_tokens, const float* __restrict__ partials, int splits,
                                                    size_t split_stride) {
#pragma clang fp contract(off)
    __shared__ float scratch[4];
    const int t = blockIdx.x;
    const size_t row = static_cast<size_t>(t) * dim;
    if (t >= n_tokens) {
        for (int i = threadIdx.x; i < dim; i += blockDim.x) {
            hi[row + i] = static_cast<half_t>(0.0f);
            lo[row + i] = static_cast<half_t>(0.0f);
        }
        return;
    }
    float ss = 0.0f;
    for (int i = 4 * threadIdx.x; i < dim; i += 4 * blockDim.x) {
        floatx4 v = *reinterpret_cast<const floatx4*>(x + row + i);
        if (splits > 0) {
            for (int z = 0; z < splits; ++z) {
                const floatx4 a = *reinterpret_cast<const floatx4*>(partials + z * split_stride + row + i);
                v = floatx4{v[0] + a[0], v[1] + a[1], v[2] + a[2], v[3] + a[3]};
            }
            *reinterpret_cast<floatx4*>(x + row + i) = v;
        }
        ss += v[0] * v[0];
        ss += v[1] * v[1];
        ss += v[2] * v[2];
        ss += v[3] * v[3];
    }
    ss = block_sum256(ss, scratch);
    ss /= static_cast<float>(dim);
    ss += 1e-5f;
    const float scale = 1.0f / sqrtf(ss);
    for (int i = 4 * threadIdx.x; i < dim; i += 4 * blockDim.x) {
        const floatx4 v = *reinterpret_cast<const floatx4*>(x + row + i);
        const floatx4 gn = *reinterpret_cast<const floatx4*>(gain + i);
#pragma unroll
        for (int e = 0; e < 4; ++e) split_store(hi, lo, row + i + e, v[e] * scale * gn[e]);
    }
}

// The same with a workgroup per row (dim = 1024 kPer) and the number of partial products known to
// the compiler: a thread's kPer x (1 + kSplits) loads are all requested before the first is used, so
// a row costs one round trip to memory and is read once.  Residual sum in the same order; the sum
// of squares runs over a thread's elements in order, across the lanes, then over the four
// wavefronts as (0 + 1) + (2 + 3).
template <int kPer, int kSplits>
__global__ __launch_bounds__(256) void k_norm_split_wide(float* __restrict__ x, const float* __restrict__ gain,
                                                         half_t* __restrict__ hi, half_t* __restrict__ lo, int n_tokens,
                                                         const float* __restrict__ partials, size_t split_stride) {
#pragma clang fp contract(off)
    constexpr int kDim = 1024 * kPer;
    __shared__ float scratch[4];
    typedef _Float16 half4_t __attribute__((ext_vector_type(4)));
    const int t = blockIdx.x;
    const size_t row = static_cast<size_t>(t) * kDim;
    const int first = 4 * threadIdx.x;
    if (t >= n_tokens) {
        const half4_t zero = {static_cast<half_t>(0.0f), static_cast<half_t>(0.0f), static_cast<half_t>(0.0f), static_cast<half_t>(0.0f)};
#pragma unroll
        for (int c = 0; c < kPer; ++c) {
            *reinterpret_cast<half4_t*>(hi + row + 1024 * c + first) = zero;
            if (lo != nullptr) *reinterpret_cast<half4_t*>(lo + row + 1024 * c + first) = zero;
        }
        return;
    }
    floatx4 v[kPer], a[kSplits > 0 ? kSplits : 1][kPer], gn[kPer];
#pragma unroll
    for (int c = 0; c < kPer; ++c) v[c] = *reinterpret_cast<const floatx4*>(x + row + 1024 * c + first);
#pragma unroll
    for (int z = 0; z < kSplits; ++z)
#pragma unroll
        for (int c = 0; c < kPer; ++c) a[z][c] = *reinterpret_cast<const floatx4*>(partials + z * split_stride + row + 1024 * c + first);
#pragma unroll
    for (int c = 0; c < kPer; ++c) gn[c] = *reinterpret_cast<const floatx4*>(gain + 1024 * c + first);
    if (kSplits > 0) {
#pragma unroll
        for (int c = 0; c < kPer; ++c) {
#pragma unroll
            for (int z = 0; z < kSplits; ++z)
                v[c] = floatx4{v[c][0] + a[z][c][0], v[c][1] + a[z][c][1], v[c][2] + a[z][c][2], v[c][3] + a[z][c][3]};
            *reinterpret_cast<floatx4*>(x + row + 1024 * c + first) = v[c];
        }
    }
    float ss = 0.0f;
#pragma unroll
    for (int c = 0; c < kPer; ++c) {
        ss += v[c][0] * v[c][0];
        ss += v[c][1] * v[c][1];
        ss += v[c][2] * v[c][2];
        ss += v[c][3] * v[c][3];
    }
    ss = block_sum256(ss, scratch);
    ss /= static_cast<float>(kDim);
    ss += 1e-5f;
    const float scale = 1.0f / sqrtf(ss);
#pragma unroll
    for (int c = 0; c < kPer; ++c) {
        half4_t h, l;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const float y = v[c][e] * scale * gn[c][e];
            h[e] = static_cast<half_t>(y);
            l[e] = static_cast<half_t>(y - static_cast<float>(h[e]));
        }
        *reinterpret_cast<half4_t*>(hi + row + 1024 * c + first) = h;
        if (lo != nullptr) *reinterpret_cast<half4_t*>(lo + row + 1024 * c + first) = l;  // (null: nobody reads the remainders)
    }
}

// RoPE on q and k of token t (ops.cpp:34-54), q kept in fp32, k and v written to the
// caches as binary16 at position pos0 + t (model.cpp:171-176).  With kSplits > 1, qs/ks/vs are the
// first of that many partial products, split_stride floats apart, and are summed in order here;
// q receives the rotated sum either way.  Grid (workgroups to a row of q, k and v, tokens): a thread has
// two pairs (16-byte loads and stores; dim, kv_dim and the head size are multiples of 4) and requests
// all its parts before it uses the first, one round trip to memory.
template <int kSplits>
__global__ __launch_bounds__(256) void k_rope_scatter(float* q, const float* qs, const float* __restrict__ ks,
                                                      const float* __restrict__ vs, const float2* __restrict__ rope,
                                                      uint16_t* __restrict__ key_cache, uint16_t* __restrict__ value_cache,
                                                      int layer, int pos0, int dim, int kv_dim, int hs, int seq_len,
                                                      size_t split_stride) {
#pragma clang fp contract(off)
    const int t = blockIdx.y, pos = pos0 + t;
    const int column = 4 * static_cast<int>(blockIdx.x * blockDim.x + threadIdx.x);
    if (column >= dim + 2 * kv_dim) return;
    const bool is_q = column < dim, is_v = column >= dim + kv_dim;
    const int i = is_q ? column : (is_v ? column - dim - kv_dim : column - dim);
    const size_t at = static_cast<size_t>(t) * (is_q ? dim : kv_dim) + i;
    const float* from = (is_q ? qs : (is_v ? vs : ks)) + at;
    const int head = i / hs, within = i - head * hs;
    floatx4 part[kSplits];
#pragma unroll
    for (int z = 0; z < kSplits; ++z) part[z] = *reinterpret_cast<const floatx4*>(from + z * split_stride);
    // (cos, sin) of two pairs
    const floatx4 cs = *reinterpret_cast<const floatx4*>(rope + static_cast<size_t>(pos) * (hs / 2) + (within >> 1));
    floatx4 v = part[0];
#pragma unroll
    for (int z = 1; z < kSplits; ++z) v = floatx4{v[0] + part[z][0], v[1] + part[z][1], v[2] + part[z][2], v[3] + part[z][3]};
    if (!is_v) v = floatx4{v[0] * cs[0] - v[1] * cs[1], v[0] * cs[1] + v[1] * cs[0], v[2] * cs[2] - v[3] * cs[3], v[2] * cs[3] + v[3] * cs[2]};
    if (is_q) {
        *reinterpret_cast<floatx4*>(q + at) = v;
        return;
    }
    typedef uint16_t ushort4_t __attribute__((ext_vector_type(4)));
    uint16_t* cache = is_v ? value_cache : key_cache;
    *reinterpret_cast<ushort4_t*>(cache + static_cast<size_t>(layer) * kv_dim * seq_len + static_cast<size_t>(head) * seq_len * hs +
                                  static_cast<size_t>(pos) * hs + within) =
        ushort4_t{f32_to_f16_bits(v[0]), f32_to_f16_bits(v[1]), f32_to_f16_bits(v[2]), f32_to_f16_bits(v[3])};
}

// (hi, lo)[t][u] = (g * sigmoid(g)) * up (ops.cpp:78-87); rows t >= n_tokens are zero.
__global__ __launch_bounds__(256) void k_swiglu_split(const float* __restrict__ gate, const float* __restrict__ up,
                                                      half_t* __restrict__ hi, half_t* __restrict__ lo, int hidden,
                                                      int n_tokens) {
#pragma clang fp contract(off)
    const int t = blockIdx.y;
    const int u = blockIdx.x * blockDim.x + threadIdx.x;
    if (u >= hidden) return;
    const size_t at = static_cast<size_t>(t) * hidden + u;
    float out = 0.0f;
    if (t < n_tokens) {
        const float g = gate[at];
        const float sigma = 1.0f / (1.0f + expf(-g));
        out = (g * sigma) * up[at];
    }
    split_store(hi, lo, at, out);
}

// ---------------------------------------------------------------------------
// GEMM on the matrix cores: Y[t][f] (+)= sum_k W[f][k] * (Xh[t][k] + Xl[t][k])
// ---------------------------------------------------------------------------
//
// W is [n][K] binary16 row-major (a weight matrix as stored), Xh/Xl are [T][K]
// binary16 row-major, Y is [T][ldy] fp32.  n % 128 == 0, T % 128 == 0, K % 32 == 0.
// A workgroup of four wavefronts owns a square tile of 128 x 128 (kSub = 2: each wavefront
// a 64 x 64 quarter = 2 x 2 MFMA tiles of 32 x 32) or of 64 x 64 (kSub = 1) features x tokens;
// the smaller tile is used when the larger one would leave compute units without a workgroup.  Both operands have k as their
// contiguous dimension, so a lane reads its 8 k-values of a fragment row as one
// 16-byte load (the two halves of the wavefront take the two halves of a 16-wide
// k-step); the weight fragment is the A operand, the activations the B operand, and
// a lane ends up holding, for ONE token, 4 runs of 4 consecutive features per tile.
template <bool kAccumulate, int kSub>
__global__ __launch_bounds__(256) void k_gemm(const half_t* __restrict__ w, const half_t* __restrict__ xh,
                                              const half_t* __restrict__ xl, float* __restrict__ y, int K, int ldy) {
    const int lane = lane_id();
    const int wave = wave_index();
    constexpr int kWaveTile = 32 * kSub;  // a wavefront's square of the workgroup's (2 * kWaveTile)^2 tile
    const int f0 = blockIdx.x * (2 * kWaveTile) + (wave & 1) * kWaveTile;
    const int t0 = blockIdx.y * (2 * kWaveTile) + (wave >> 1) * kWaveTile;
    const int r = lane & 31, g = lane >> 5;
    const half_t* wrow[kSub];
    const half_t* hrow[kSub];
    const half_t* lrow[kSub];
#pragma unroll
    for (int i = 0; i < kSub; ++i) {
        wrow[i] = w + static_cast<size_t>(f0 + 32 * i + r) * K + 8 * g;
        hrow[i] = xh + static_cast<size_t>(t0 + 32 * i + r) * K + 8 * g;
        lrow[i] = xl + static_cast<size_t>(t0 + 32 * i + r) * K + 8 * g;
    }
    floatx16 acc[kSub][kSub];
#pragma unroll
    for (int i = 0; i < kSub; ++i)
#pragma unroll
        for (int j = 0; j < kSub; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.0f;

    // Two k-steps (32 columns) per trip: a lane's two 16-byte pieces of a row are 32 bytes apart, and a
    // row's 128-byte line is used up in two trips while it is still in the cache.  The fragments of the
    // next trip are requested before this trip's products are issued.
    struct Frags {
        half8_t a[2][kSub], bh[2][kSub], bl[2][kSub];
    };
    auto fetch = [&](Frags& f, int k0) {
#pragma unroll
        for (int s = 0; s < 2; ++s)
#pragma unroll
            for (int i = 0; i < kSub; ++i) {
                f.a[s][i] = *reinterpret_cast<const half8_t*>(wrow[i] + k0 + 16 * s);
                f.bh[s][i] = *reinterpret_cast<const half8_t*>(hrow[i] + k0 + 16 * s);
                f.bl[s][i] = *reinterpret_cast<const half8_t*>(lrow[i] + k0 + 16 * s);
            }
    };
    auto multiply = [&](const Frags& f) {
#pragma unroll
        for (int s = 0; s < 2; ++s)
#pragma unroll
            for (int i = 0; i < kSub; ++i)
#pragma unroll
                for (int j = 0; j < kSub; ++j) {
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(f.a[s][i], f.bh[s][j], acc[i][j], 0, 0, 0);
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(f.a[s][i], f.bl[s][j], acc[i][j], 0, 0, 0);
                }
    };
    Frags cur, nxt;
    fetch(cur, 0);
    for (int k0 = 32; k0 < K; k0 += 32) {
        fetch(nxt, k0);
        multiply(cur);
        cur = nxt;
    }
    multiply(cur);
    // D[m][n]: lane holds column n = lane % 32 (a token) and rows m = 8 * (e / 4) + 4 * (lane / 32) + e % 4 (features)
#pragma unroll
    for (int i = 0; i < kSub; ++i)
#pragma unroll
        for (int j = 0; j < kSub; ++j) {
            float* row = y + static_cast<size_t>(t0 + 32 * j + r) * ldy + f0 + 32 * i + 4 * g;
#pragma unroll
            for (int e4 = 0; e4 < 4; ++e4) {
                floatx4* dst = reinterpret_cast<floatx4*>(row + 8 * e4);
                floatx4 v = floatx4{acc[i][j][4 * e4], acc[i][j][4 * e4 + 1], acc[i][j][4 * e4 + 2], acc[i][j][4 * e4 + 3]};
                if constexpr (kAccumulate) {
                    const floatx4 old = *dst;
                    v = floatx4{old[0] + v[0], old[1] + v[1], old[2] + v[2], old[3] + v[3]};
                }
                *dst = v;
            }
        }
}

// The same product as a pipeline of LDS stages filled by the memory system itself.
//
// A workgroup is eight wavefronts: four that multiply and four that only request data.  A request
// instruction holds its wavefront until the compute unit's memory pipeline has taken it (64 bytes
// a cycle: a trip's 64 KiB are 1000 cycles of that), and a wavefront that issues MFMAs cannot
// issue them while it is held, so the requests go out from wavefronts with nothing else to do;
// a SIMD runs one of each kind.
//
// The four multiplying wavefronts (2 x 2) own a tile of 64 kFi features x 64 kTj tokens; a wavefront
// owns 32 kFi x 32 kTj of it (2 kFi x 2 kTj MFMA tiles of 16 x 16: the weight side is the longer one, because the
// activations come twice, as head and remainder, and every fragment is read from LDS once per
// wavefront that uses it).  What bounds a full tile is the device's power, so the products are
// v_mfma_f32_16x16x32_f16, remainder right behind head in the same accumulator: 32 x 32 x 16 needs a lower clock for the same
// work (the exact mode's W1+W3, 512 ids: 1B shape 69 -> 63 us, 8B 252 -> 224; of 2048 ids of the 1B shape 260 -> 236, W2 127 ->
// 112; the fast mode, half of it data, 2 to 5 %).  A trip covers 64 columns, a whole cache line of every row: L2 gives a compute
// unit 100 bytes a nanosecond in requests of whole lines and 70 in halves of lines (256 workgroups of eight wavefronts that do
// nothing but request rows 4 KiB apart from 256 KiB to 2 MiB; contiguous, 105 to 111).  The rows of the three operand tiles lie
// one after the other in a stage of LDS, and a requesting wavefront fills 1 KiB of it
// with one global_load_lds_dwordx4 (lane i -> 16 bytes at M0 + 16 i): no registers are staged
// and nothing waits for the data but the s_waitcnt ahead of the trip that multiplies it.  As
// many stages as 160 KiB hold, five at most.  Of 256 x 128 tiles in the exact mode a stage would be 64 KiB, two of them too few:
// there a trip's weight rows and its token rows are halves of 32 KiB that come and go by themselves, five of them; the weights
// have two trips to arrive in, the tokens one.  (W1+W3 of 512 ids of the 1B shape, with trips of 32 columns in five stages
// and so: exact mode 67.9 -> 63.3 us, a prefill 2.33 -> 2.27 ms; fast mode, in three whole stages, 1.87 -> 1.76.)
//
// LDS banks: a fragment read takes 16 bytes per lane from 16 consecutive rows; with rows of 128
// bytes every second row starts in the same bank, so the 16-byte pieces of row r
// are stored in the order piece ^ ((r >> 1) & 7): 16 consecutive lanes then
// cover all 64 banks once.  The permutation is applied on the way in, by the address each lane
// requests.
//
// The requests are inline assembly: written with the builtin, every LDS read of the loop would
// wait for all outstanding requests (they may alias), which is the pipeline's whole depth.
//
// kMode 0 stores the tile, 1 adds it to y, 2 is the feed-forward pair: the tile's weight rows are
// 32 kFi features of W1 (the wavefront's first kFi MFMA tiles) and the same features of W3
// (its last kFi), and what is stored is (g * sigmoid(g)) * up (ops.cpp:78-87), split into
// binary16 head and remainder as the next product wants it.
struct PipeJob {
    const half_t* w[3];
    float* y[3];
    int ldy[3];
    int first_tile[3];  // first feature tile of matrix i (first_tile[0] = 0); unused entries = INT_MAX
    const half_t* xh;
    const half_t* xl;
    int K;      // row length of w and x
    int k_len;  // columns a workgroup multiplies: split z covers [z * k_len, (z + 1) * k_len) and writes y + z * split_stride
    size_t split_stride;
    int feature_tiles, token_tiles, groups;  // groups = feature_tiles * splits
    int band;                                // k_gemm_pipe: token tiles a die's workgroups take at a time; divides token_tiles
    half_t* out_hi;                          // kMode 2: [tokens][out_ld]
    half_t* out_lo;
    int out_ld;
    int live, each;  // tokens there are; k_gemm_pipe, kRagged: tokens to a tile (a multiple of 32)
    int rows;        // k_gemm_block: rows of x and of the output, a multiple of 32
};

constexpr int kPipeTripK = 64;  // columns per trip; K must be a multiple

// (kLo: the activations' remainder tile travels and is multiplied too; without it a stage is a third smaller)
template <int kFi, int kTj, bool kLo = true>
struct PipeShape {
    static constexpr int kRowBytes = 2 * kPipeTripK;
    static constexpr int kRowsA = 64 * kFi, kRowsB = 64 * kTj, kRows = kRowsA + (kLo ? 2 : 1) * kRowsB;
    static constexpr int kStageBytes = kRows * kRowBytes;
    // (where a trip's rows of weights and of tokens are 32 KiB each, they come and go by themselves: five such halves)
    static constexpr bool kHalves = kStageBytes == 65536 && kRowsA == kRows / 2;
    static constexpr int kStages = (160 * 1024) / kStageBytes > 5 ? 5 : (160 * 1024) / kStageBytes;
    static constexpr int kLoads = kStageBytes / 4096;  // requests of 1 KiB per wavefront and stage
    static constexpr int kLdsBytes = kHalves ? 5 * 32768 : kStages * kStageBytes;
};

template <int kCount>
__device__ __forceinline__ void wait_requests() {
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(kCount) : "memory");
}

typedef _Float16 half4_pf_t __attribute__((ext_vector_type(4)));

// (hi, lo) = SwiGLU of four (gate, up) pairs, ops.cpp:78-87
__device__ __forceinline__ void swiglu_split4(half4_pf_t& hi, half4_pf_t& lo, const float* g, const float* u) {
#pragma clang fp contract(off)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const float sigma = 1.0f / (1.0f + expf(-g[e]));  // (hardware exp and reciprocal here: 0.4 % of a prefill)
        const float v = (g[e] * sigma) * u[e];
        hi[e] = static_cast<half_t>(v);
        lo[e] = static_cast<half_t>(v - static_cast<float>(hi[e]));
    }
}

// A wavefront's sums on their way out.  D[m][n]: a lane holds column n = lane % 16 (a token) and rows m = 4 (lane / 16) + e
// (features): stored from there, an instruction would write 16 bytes or 8 to each of 16 rows of the output.  The tiles
// therefore pass through LDS, [token][feature], and leave as whole lines, eight lanes to a token's row.  `room`: kLeaveBytes that are the
// wavefront's own; its LDS accesses are served in order, so no barrier is needed between a tile's writes, its reads and
// the next tile's writes.  t0: the wavefront's first token, f_base: the workgroup's first feature, wf: the wavefront's
// place along the features; only the first live_tiles token tiles are stored.
constexpr int kLeaveBytes = 32 * 36 * 4;
template <int kMode, bool kLo, int kI, int kJ>
__device__ __forceinline__ void leave(const floatx4 (&acc)[kI][kJ], char* room, const PipeJob& job, int which, int split, int t0, int live_tiles,
                                      int f_base, int wf) {
    const int lane = lane_id();
    if constexpr (kMode == 2) {
        static_assert(kI % 2 == 0, "a wavefront's gate and up tiles: as many of each");
        constexpr int kPairs = kI / 2, kWide = 16 * kPairs;  // features of the wavefront's output
        constexpr int kPitch = kWide + 8;                    // binary16 per token row of the transposed tile, padding included
        constexpr int kLanes = kWide / 8, kRowsAtOnce = 64 / kLanes;
        static_assert(16 * kPitch * 2 <= kLeaveBytes, "room");
        const int part = lane % kLanes, row_of = lane / kLanes;
        half_t* tile = reinterpret_cast<half_t*>(room);
#pragma unroll
        for (int j = 0; j < kJ; ++j) {
            if (j >= live_tiles) break;
            half4_pf_t h[kPairs], l[kPairs];
#pragma unroll
            for (int i = 0; i < kPairs; ++i) {
                const float gate[4] = {acc[i][j][0], acc[i][j][1], acc[i][j][2], acc[i][j][3]};
                const float up[4] = {acc[i + kPairs][j][0], acc[i + kPairs][j][1], acc[i + kPairs][j][2], acc[i + kPairs][j][3]};
                swiglu_split4(h[i], l[i], gate, up);
            }
            const size_t at = static_cast<size_t>(t0 + 16 * j) * job.out_ld + f_base + wf * kWide + 8 * part;
            // (without kLo the next GEMM reads no remainders either)
#pragma unroll
            for (int which_half = 0; which_half < (kLo ? 2 : 1); ++which_half) {
#pragma unroll
                for (int i = 0; i < kPairs; ++i)
                    *reinterpret_cast<half4_pf_t*>(tile + (lane & 15) * kPitch + 16 * i + 4 * (lane >> 4)) = which_half == 0 ? h[i] : l[i];
                half_t* out = which_half == 0 ? job.out_hi : job.out_lo;
#pragma unroll
                for (int pass = 0; pass < 16 / kRowsAtOnce; ++pass) {
                    const int n = kRowsAtOnce * pass + row_of;
                    *reinterpret_cast<half8_t*>(out + at + static_cast<size_t>(n) * job.out_ld) =
                        *reinterpret_cast<const half8_t*>(tile + n * kPitch + 8 * part);
                }
            }
        }
    } else {
        constexpr int kPitch = 36;  // floats per token row of the transposed tile: 32 features + padding
        const int part8 = lane & 7, row8 = lane >> 3;
        float* tile = reinterpret_cast<float*>(room);
        float* __restrict__ y = (which == 2 ? job.y[2] : (which == 1 ? job.y[1] : job.y[0])) + static_cast<size_t>(split) * job.split_stride;
        const int ldy = which == 2 ? job.ldy[2] : (which == 1 ? job.ldy[1] : job.ldy[0]);
#pragma unroll
        for (int j = 0; j < kJ; j += 2) {
            if (j >= live_tiles) break;
#pragma unroll
            for (int i = 0; i < kI; i += 2) {
#pragma unroll
                for (int jj = 0; jj < 2; ++jj)
#pragma unroll
                    for (int ii = 0; ii < 2; ++ii)
                        *reinterpret_cast<floatx4*>(tile + (16 * jj + (lane & 15)) * kPitch + 16 * ii + 4 * (lane >> 4)) = acc[i + ii][j + jj];
                float* first = y + static_cast<size_t>(t0 + 16 * j) * ldy + f_base + wf * 16 * kI + 16 * i + 4 * part8;
#pragma unroll
                for (int pass = 0; pass < 4; ++pass) {
                    const int n = 8 * pass + row8;
                    floatx4* out = reinterpret_cast<floatx4*>(first + static_cast<size_t>(n) * ldy);
                    floatx4 v = *reinterpret_cast<const floatx4*>(tile + n * kPitch + 4 * part8);
                    if constexpr (kMode == 1) {
                        const floatx4 old = *out;
                        v = floatx4{old[0] + v[0], old[1] + v[1], old[2] + v[2], old[3] + v[3]};
                    }
                    *out = v;
                }
            }
        }
    }
}

template <int kFi, int kTj, int kMode, bool kLo, bool kRagged>
__global__ __launch_bounds__(512) void k_gemm_pipe(PipeJob job) {
    typedef PipeShape<kFi, kTj, kLo> Shape;
    constexpr int kRowsA = Shape::kRowsA, kRowsB = Shape::kRowsB, kStages = Shape::kStages, kLoads = Shape::kLoads;
    constexpr int kStageBytes = Shape::kStageBytes, kRowBytes = Shape::kRowBytes;
    constexpr bool kHalves = Shape::kHalves;
    constexpr int kSteps = kPipeTripK / 32;  // k-steps per trip
    constexpr int kPieces = kPipeTripK / 8;  // 16-byte pieces of a row
    extern __shared__ __align__(1024) char pipe_lds[];
    const int lane = lane_id();
    const int wave_of_8 = __builtin_amdgcn_readfirstlane(wave_index());
    const bool requester = wave_of_8 >= 4;
    const int wave = wave_of_8 & 3;  // which quarter of the tile (multiplying) or of the requests (requesting)
    // Workgroups are handed to the eight dies in turn: those that share a weight tile (same features
    // and columns, other tokens) get numbers that are equal modulo 8, so the tile crosses one die's L2.
    const int id = static_cast<int>(blockIdx.x), die = id & 7, within = id >> 3;
    // Of many token tiles, job.band at a time: a die's 32 compute units then hold, at 16 token tiles, eight weight tiles and
    // four activation tiles at once instead of two and 16.  (band divides token_tiles.)
    const int per_band = ((job.groups + 7) >> 3) * job.band, band = within / per_band, in_band = within - band * per_band;
    const int group = (in_band / job.band) * 8 + die;
    if (group >= job.groups) return;
    const int token_tile = band * job.band + in_band % job.band;
    const int tile_all = group % job.feature_tiles, split = group / job.feature_tiles;
    const int which = tile_all >= job.first_tile[2] ? 2 : (tile_all >= job.first_tile[1] ? 1 : 0);
    const int tile_x = tile_all - (which == 2 ? job.first_tile[2] : (which == 1 ? job.first_tile[1] : 0));
    const half_t* __restrict__ w = which == 2 ? job.w[2] : (which == 1 ? job.w[1] : job.w[0]);
    const int K = job.K, k_first = split * job.k_len;
    const int wf = wave & 1, wt = wave >> 1;
    constexpr int kFeaturesPerTile = kMode == 2 ? 32 * kFi : 64 * kFi;
    const int f_base = tile_x * kFeaturesPerTile, t_base = token_tile * (kRagged ? job.each : kRowsB);

    // (a row past the tile's: any, nobody multiplies it)
    auto row_of = [&](int row) { return kRagged && row >= job.each ? job.each - 1 : row; };
    // what each lane requests: request q of this wavefront fills 1 KiB = rows (64 / kPieces) (wave + 4 q) .. of a stage
    const char* src[kLoads];
#pragma unroll
    for (int q = 0; q < kLoads; ++q) {
        const int row = (64 / kPieces) * (wave + 4 * q) + lane / kPieces;
        const int piece = (lane % kPieces) ^ ((row >> 1) & (kPieces - 1));
        const half_t* from;
        if (row < kRowsA) {
            if constexpr (kMode == 2) {
                const int wave_rows = 32 * kFi, half_rows = 16 * kFi;
                const int owner = row / wave_rows, rem = row % wave_rows;
                const half_t* matrix = rem >= half_rows ? job.w[1] : job.w[0];
                from = matrix + static_cast<size_t>(f_base + owner * half_rows + rem % half_rows) * K;
            } else {
                from = w + static_cast<size_t>(f_base + row) * K;
            }
        } else if (!kLo || row < kRowsA + kRowsB) {
            from = job.xh + static_cast<size_t>(t_base + row_of(row - kRowsA)) * K;
        } else {
            from = job.xl + static_cast<size_t>(t_base + row_of(row - kRowsA - kRowsB)) * K;
        }
        src[q] = reinterpret_cast<const char*>(from + k_first) + 16 * piece;
    }
    const unsigned lds_base = static_cast<unsigned>(reinterpret_cast<uintptr_t>(
        (__attribute__((address_space(3))) char*)pipe_lds));
    const int trips = job.k_len / kPipeTripK;
    // (tile_columns: columns of 32 tokens that the tile has; the requests of the others are not made)
    constexpr int kWeightLoads = kRowsA / (64 / kPieces) / 4, kTileColumns = 2 * kTj;
    auto made = [&](int q, int tile_columns) { return q < kWeightLoads || (q - kWeightLoads) % kTileColumns < tile_columns; };
    auto request = [&](int trip, auto tile_columns) {
        const unsigned at = __builtin_amdgcn_readfirstlane(lds_base + (trip % kStages) * kStageBytes + wave * 1024);
        const int column = __builtin_amdgcn_readfirstlane(trip * kRowBytes);
#pragma unroll
        for (int q = 0; q < kLoads; ++q)
            if (made(q, tile_columns)) {
                const char* from = src[q] + column;
                const unsigned to = at + q * 4096;
                asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off\n" ::"v"(from), "s"(to) : "memory");
            }
    };
    // kHalves: half u is the weight rows of trip u / 2 (even) or its token rows
    auto request_half = [&](int u, auto odd, auto tile_columns) {
        const unsigned at = __builtin_amdgcn_readfirstlane(lds_base + (u % 5) * 32768 + wave * 1024);
        const int column = __builtin_amdgcn_readfirstlane((u >> 1) * kRowBytes);
#pragma unroll
        for (int q = odd * kWeightLoads; q < (odd ? kLoads : kWeightLoads); ++q)
            if (made(q, tile_columns)) {
                const char* from = src[q] + column;
                const unsigned to = at + (q - odd * kWeightLoads) * 4096;
                asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off\n" ::"v"(from), "s"(to) : "memory");
            }
    };
    // where each lane reads its fragments: row lane % 16 of an MFMA tile, piece 4 s + lane / 16 of k-step s
    int a_off[kSteps], b_off[kSteps];
#pragma unroll
    for (int s = 0; s < kSteps; ++s) {
        const int row = lane & 15, piece = (4 * s + (lane >> 4)) ^ ((row >> 1) & (kPieces - 1));
        a_off[s] = (wf * 32 * kFi + row) * kRowBytes + 16 * piece;
        b_off[s] = ((kHalves ? 0 : kRowsA) + wt * 32 * kTj + row) * kRowBytes + 16 * piece;
    }

    constexpr int kI = 2 * kFi, kJ = 2 * kTj;  // MFMA tiles of the wavefront
    floatx4 acc[kI][kJ];
#pragma unroll
    for (int i = 0; i < kI; ++i)
#pragma unroll
        for (int j = 0; j < kJ; ++j) acc[i][j] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};

    struct Tokens {
        half8_t h[kJ], l[kJ];
    };
    half8_t a[kI];
    auto read_tokens = [&](Tokens& f, int trip, int s, int j) {
        const char* stage = pipe_lds + (kHalves ? (2 * trip + 1) % 5 * 32768 : (trip % kStages) * kStageBytes);
        f.h[j] = *reinterpret_cast<const half8_t*>(stage + b_off[s] + j * 16 * kRowBytes);
        if constexpr (kLo) f.l[j] = *reinterpret_cast<const half8_t*>(stage + b_off[s] + (kRowsB + j * 16) * kRowBytes);
    };
    auto read_weights = [&](int trip, int s, int i) {
        const char* stage = pipe_lds + (kHalves ? 2 * trip % 5 * 32768 : (trip % kStages) * kStageBytes);
        a[i] = *reinterpret_cast<const half8_t*>(stage + a_off[s] + i * 16 * kRowBytes);
    };
    // (one weight tile's MFMAs of a k-step)
    auto multiply_row = [&](const Tokens& f, int i, auto columns) {
#pragma unroll
        for (int j = 0; j < 2 * columns; ++j) {
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[i], f.h[j], acc[i][j], 0, 0, 0);
            if constexpr (kLo) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[i], f.l[j], acc[i][j], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    // (requesting wavefronts) wait until the requests of `trip` have landed: those of later trips, at
    // most kStages - 2 of them, may be in flight
    auto landed = [&](int trip, int trips, auto tile_columns) {
        constexpr int kMade = kLoads - (kLo ? 2 : 1) * (kTileColumns - decltype(tile_columns)::value);
        const int later = trips - 1 - trip;
        if (kStages > 2 && later >= kStages - 2) wait_requests<(kStages - 2) * kMade>();
        else wait_requests<0>();
    };
    // One barrier per trip, inside the last k-step of the trip before: the requesting wavefronts
    // arrive when the trip's data has landed, the multiplying ones when they hold the last
    // fragments of the trip before in registers, which frees that trip's stage for the requests of
    // trip t + kStages.
    const int tile_end = kRagged ? min(job.live, t_base + job.each) : t_base + kRowsB;
    auto feed = [&](auto tile_columns) {
        if constexpr (kHalves) {
            // Weights, which may come from memory, have two trips to arrive in, tokens, which are in L2, one.
            constexpr int kTokenLoads = (kLo ? 2 : 1) * decltype(tile_columns)::value;
            constexpr std::integral_constant<int, 0> weights{};
            constexpr std::integral_constant<int, 1> tokens{};
            request_half(0, weights, tile_columns);
            request_half(1, tokens, tile_columns);
            if (trips > 1) {
                request_half(2, weights, tile_columns);
                request_half(3, tokens, tile_columns);
            }
            if (trips > 2) {
                request_half(4, weights, tile_columns);
                wait_requests<2 * kWeightLoads + kTokenLoads>();
            } else if (trips > 1) {
                wait_requests<kWeightLoads + kTokenLoads>();
            } else {
                wait_requests<0>();
            }
            __syncthreads();
            for (int t = 0; t < trips; ++t) {
                if (t + 2 < trips) wait_requests<kWeightLoads>();  // (those of trip t + 2)
                else wait_requests<0>();
                __syncthreads();
                if (t + 2 < trips) request_half(2 * t + 5, tokens, tile_columns);
                if (t + 3 < trips) request_half(2 * t + 6, weights, tile_columns);
            }
            return;
        }
#pragma unroll
        for (int t = 0; t < kStages - 1; ++t)
            if (__builtin_expect(t < trips, 1)) request(t, tile_columns);
        landed(0, trips, tile_columns);
        __syncthreads();
        if (__builtin_expect(kStages - 1 < trips, 1)) request(kStages - 1, tile_columns);
        for (int t = 0; t < trips; ++t) {
            landed(t + 1, trips, tile_columns);
            __syncthreads();
            if (t + kStages < trips) request(t + kStages, tile_columns);
        }
    };
    if (requester) {
        if constexpr (kRagged) {
            static_assert(kTileColumns == 4, "columns of a tile");
            const int tile_columns = __builtin_amdgcn_readfirstlane((tile_end - t_base + 31) / 32);
            if (tile_columns >= 4) feed(std::integral_constant<int, 4>{});
            else if (tile_columns == 3) feed(std::integral_constant<int, 3>{});
            else if (tile_columns == 2) feed(std::integral_constant<int, 2>{});
            else feed(std::integral_constant<int, 1>{});
        } else {
            feed(std::integral_constant<int, kTileColumns>{});
        }
        return;
    }
    // The weight tiles of a k-step are multiplied one after the other, and each one's registers take the next k-step's
    // fragment as soon as it is done; the tokens' fragments are in two sets.  The next trip's barrier is behind the first
    // quarter of the last k-step: by then every read of this trip has long been served.
    auto walk = [&](auto columns) {
        Tokens tokens[2];
        __syncthreads();
        if (columns != 0) {
#pragma unroll
            for (int j = 0; j < 2 * columns; ++j) read_tokens(tokens[0], 0, 0, j);
#pragma unroll
            for (int i = 0; i < kI; ++i) read_weights(0, 0, i);
        }
        constexpr int kMeet = kI / 4 - 1;
        auto step = [&](const Tokens& cur, Tokens& next, int t, auto s) {
            constexpr bool last = decltype(s)::value == kSteps - 1;
            constexpr int s_next = last ? 0 : decltype(s)::value + 1;
            // (after the last trip this reads a stage nobody uses: one path through the loop)
            const int t_next = last ? t + 1 : t;
#pragma unroll
            for (int i = 0; i < kI; ++i) {
                multiply_row(cur, i, columns);
                if constexpr (last)
                    if (i == kMeet) {
                        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
                        __syncthreads();
                    }
                if (i >= kMeet && columns != 0) {
#pragma unroll
                    for (int k = i == kMeet ? 0 : i; k <= i; ++k) read_weights(t_next, s_next, k);
                    if (i < kMeet + 2)
#pragma unroll
                        for (int j = (i - kMeet) * columns; j < (i - kMeet + 1) * columns; ++j) read_tokens(next, t_next, s_next, j);
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
        };
        static_assert(kSteps == 2, "the tokens' fragments of a trip are in the two sets");
        for (int t = 0; t < trips; ++t) {
            step(tokens[0], tokens[1], t, std::integral_constant<int, 0>{});
            step(tokens[1], tokens[0], t, std::integral_constant<int, 1>{});
        }
    };
    // kRagged: columns of 32 tokens that are not the tile's, or past the last token, are neither multiplied nor stored.
    int columns = kTj;
    if constexpr (kRagged) {
        static_assert(kTj == 2, "columns of a wavefront: 0, 1 or 2");
        columns = __builtin_amdgcn_readfirstlane(max(0, min(kTj, (tile_end - t_base - wt * 32 * kTj + 31) / 32)));
        if (columns == 2) walk(std::integral_constant<int, 2>{});
        else if (columns == 1) walk(std::integral_constant<int, 1>{});
        else walk(std::integral_constant<int, 0>{});
    } else {
        walk(std::integral_constant<int, kTj>{});
    }
    // (room: the wavefront's quarter of a stage that neither the last trip nor the read past it uses)
    static_assert(kHalves ? kLeaveBytes <= 8192 : kStages >= 3 && kStageBytes / 4 >= kLeaveBytes, "room for a transposed tile per wavefront");
    char* room = pipe_lds + (kHalves ? (2 * trips + 2) % 5 * 32768 + wave * 8192 : ((trips + 1) % kStages) * kStageBytes + wave * (kStageBytes / 4));
    leave<kMode, kLo>(acc, room, job, which, split, t_base + wt * 32 * kTj, kRagged ? 2 * columns : kJ, f_base, wf);
}

// The same product in blocks of 256 features x 256 tokens, for batches that make enough of them.
//
// Eight wavefronts, two to a SIMD, all of them multiply: each owns 128 features x 64 tokens.  The two of a SIMD take turns,
// one barrier apart: while one multiplies a trip of 32 columns, the other reads its fragments of the trip from LDS and sends
// for a later one, so the matrix cores are busy but for the barriers (exact mode: 4650 clocks of the loop for 64 columns, 4096
// of them MFMAs; 72 % of the whole launch's clocks at 2048 ids of the 1B shape) and a wavefront that a request holds up holds
// nobody else.  A trip's rows are 64 bytes, their pieces in the order piece ^ ((r >> 2) & 3); kStages trips are in LDS at once.
// (By the counters half of the reads' LDS cycles are bank conflicts in that order, where k_gemm_pipe's rows of 128 bytes have
// next to none.  LDS is busy for 38 % of the launch, behind the matrix cores.)
//
// What bounds it is the device's power, not its clocks: the exact mode's launches run at 1.7 to 1.9 GHz, and what makes them
// faster is less energy to a product.  That is why a block is as large as the registers allow (from L2 a quarter fewer bytes to
// a product than 256 x 128, without the remainders a third; from LDS as many), and why the products are
// v_mfma_f32_16x16x32_f16, head and remainder one after the other into the same accumulator: of the same block, W1+W3 of 2048
// ids of the 1B shape takes 233 us in products of 32 x 32 x 16, 213 in 16 x 16 x 32, and 204 with the accumulator kept from head
// to remainder (266 in k_gemm_pipe's tiles of 256 x 128); without the remainders 134, 126 (and 160).  Fed from registers alone,
// with neither requests nor reads, the same loop takes 168 us.
constexpr int kBlock = 256;  // features and tokens of a block
template <bool kLo>
struct BlockShape {
    static constexpr int kTripK = 32, kRowBytes = 2 * kTripK;
    static constexpr int kRows = (kLo ? 3 : 2) * kBlock;
    static constexpr int kStageBytes = kRows * kRowBytes;
    static constexpr int kStages = (160 * 1024) / kStageBytes;
    static constexpr int kLoads = kRows / 128;  // requests of 1 KiB per wavefront and stage
    static constexpr int kLdsBytes = kStages * kStageBytes;
    static_assert(kStages >= 3, "stages of a workgroup");
};

template <int kMode, bool kLo>
__global__ __launch_bounds__(512, 2) void k_gemm_block(PipeJob job) {
    typedef BlockShape<kLo> Shape;
    constexpr int kStages = Shape::kStages, kLoads = Shape::kLoads, kStageBytes = Shape::kStageBytes, kRowBytes = Shape::kRowBytes;
    constexpr int kWaveF = 128, kI = kWaveF / 16, kJ = 4;
    extern __shared__ __align__(1024) char block_lds[];
    const int lane = lane_id();
    const int wave = __builtin_amdgcn_readfirstlane(wave_index());
    // (workgroups that share a weight tile on one die, job.band token tiles at a time: as in k_gemm_pipe)
    const int id = static_cast<int>(blockIdx.x), die = id & 7, within = id >> 3;
    const int per_band = ((job.groups + 7) >> 3) * job.band, band = within / per_band, in_band = within - band * per_band;
    const int group = (in_band / job.band) * 8 + die;
    if (group >= job.groups) return;
    const int token_tile = band * job.band + in_band % job.band;
    const int tile_all = group % job.feature_tiles, split = group / job.feature_tiles;
    const int which = tile_all >= job.first_tile[2] ? 2 : (tile_all >= job.first_tile[1] ? 1 : 0);
    const int tile_x = tile_all - (which == 2 ? job.first_tile[2] : (which == 1 ? job.first_tile[1] : 0));
    const half_t* __restrict__ w = which == 2 ? job.w[2] : (which == 1 ? job.w[1] : job.w[0]);
    const int K = job.K, k_first = split * job.k_len;
    const int wf = wave & 1, wt = wave >> 1;
    const bool second = wave >= 4;  // (wavefronts w and w + 4 share a SIMD)
    const int f_base = tile_x * (kMode == 2 ? kBlock / 2 : kBlock), t_base = token_tile * kBlock;

    // Request q of this wavefront fills 1 KiB of a stage: 16 rows from 16 (wave + 8 q) on, four lanes to a row's 64 bytes.  The
    // lanes' offsets from the first row are the same for all of them.  Token rows past the buffer's are its last ones again.
    const unsigned lane_off = static_cast<unsigned>(lane >> 2) * static_cast<unsigned>(2 * K) + 16u * ((lane & 3) ^ (lane >> 4));
    const char* base[kLoads];
#pragma unroll
    for (int q = 0; q < kLoads; ++q) {
        const int row = 16 * (wave + 8 * q);
        const half_t* from;
        if (row < kBlock) {
            if constexpr (kMode == 2) {
                const int owner = row / kWaveF, rem = row % kWaveF;
                from = (rem >= kWaveF / 2 ? job.w[1] : job.w[0]) + static_cast<size_t>(f_base + owner * (kWaveF / 2) + rem % (kWaveF / 2)) * K;
            } else {
                from = w + static_cast<size_t>(f_base + row) * K;
            }
        } else {
            from = (kLo && row >= 2 * kBlock ? job.xl : job.xh) + static_cast<size_t>(min(t_base + row % kBlock, job.rows - 16)) * K;
        }
        base[q] = reinterpret_cast<const char*>(from + k_first);
    }
    const unsigned lds_base = static_cast<unsigned>(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) char*)block_lds));
    const int trips = job.k_len / Shape::kTripK;
    auto request = [&](int trip, int slot) {
        const unsigned at = __builtin_amdgcn_readfirstlane(lds_base + slot * kStageBytes + wave * 1024);
        const unsigned off = lane_off + static_cast<unsigned>(trip) * kRowBytes;
        // (s_nop 4: the scalar address may have been written by a vector instruction just before)
#pragma unroll
        for (int q = 0; q < kLoads; ++q)
            asm volatile("s_mov_b32 m0, %2\n\ts_nop 4\n\tglobal_load_lds_dwordx4 %0, %1\n" ::"v"(off), "s"(base[q]), "s"(at + q * 8192) : "memory");
    };
    // `trip` has landed: of this wavefront's requests those of the kStages - 2 trips behind it may be out
    auto landed = [&](int trip) {
        if (trips - 1 - trip >= kStages - 2) wait_requests<(kStages - 2) * kLoads>();
        else wait_requests<0>();
    };
    auto meet = [] {
        __builtin_amdgcn_sched_barrier(0);
        asm volatile("s_barrier" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
    };

    // fragments: row lane % 16 of a 16-row tile, the 16-byte piece lane / 16 of the trip's 64 bytes
    const int read_off = (lane & 15) * kRowBytes + 16 * ((lane >> 4) ^ ((lane >> 2) & 3));
    floatx4 acc[kI][kJ];
#pragma unroll
    for (int i = 0; i < kI; ++i)
#pragma unroll
        for (int j = 0; j < kJ; ++j) acc[i][j] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
    half8_t a[kI], bh[kJ], bl[kJ];
    auto read = [&](int slot) {
        const char* rows_a = block_lds + slot * kStageBytes + wf * kWaveF * kRowBytes + read_off;
        const char* rows_b = block_lds + slot * kStageBytes + (kBlock + wt * 64) * kRowBytes + read_off;
#pragma unroll
        for (int j = 0; j < kJ; ++j) {
            bh[j] = *reinterpret_cast<const half8_t*>(rows_b + 16 * j * kRowBytes);
            if constexpr (kLo) bl[j] = *reinterpret_cast<const half8_t*>(rows_b + (kBlock + 16 * j) * kRowBytes);
        }
#pragma unroll
        for (int i = 0; i < kI; ++i) a[i] = *reinterpret_cast<const half8_t*>(rows_a + 16 * i * kRowBytes);
    };
    auto multiply = [&]() {
#pragma unroll
        for (int j = 0; j < kJ; ++j)
#pragma unroll
            for (int i = 0; i < kI; ++i) {
                acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[i], bh[j], acc[i][j], 0, 0, 0);
                if constexpr (kLo) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[i], bl[j], acc[i][j], 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);  // (in this order)
            }
    };
    // A trip is read by the first group in one turn and by the second in the next; what is sent for into its stage, behind the
    // second one's turn, has kStages - 1 trips less a turn to arrive.  It must have before the first group's read of it: every
    // wavefront waits for its own requests ahead of the barrier before that.
#pragma unroll
    for (int t = 0; t < kStages - 1; ++t)
        if (t < trips) request(t, t);
    landed(0);
    meet();
    if (second) meet();
    int slot = 0, into = kStages - 1;
    const bool idle = t_base + 64 * wt >= job.live;  // (none of this wavefront's tokens is one: it only sends for rows)
    for (int t = 0; t < trips; ++t) {
        if (!idle) read(slot);
        if (t + kStages - 1 < trips) request(t + kStages - 1, into);
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        if (second) landed(t + 1);
        meet();
        if (!idle) multiply();
        if (!second) landed(t + 1);
        meet();
        into = slot;
        slot = slot + 1 == kStages ? 0 : slot + 1;
    }
    if (!second) meet();
    if (idle) return;
    // (the stages are free)
    static_assert(Shape::kLdsBytes >= 8 * kLeaveBytes, "room for a transposed tile per wavefront");
    leave<kMode, kLo>(acc, block_lds + wave * kLeaveBytes, job, which, split, t_base + 64 * wt, min(kJ, (job.rows - t_base - 64 * wt) / 16), f_base, wf);
}

// The same product for a batch of few tokens, where the weights are the traffic and the tiles above would leave most
// of the device without a workgroup.
//
// A tile is 32 kFi features x 32 kTj tokens (kTj: the whole batch up to 128 tokens), so that a matrix of a few thousand
// rows still makes a workgroup per compute unit.  Such a tile is too small to be cut among four wavefronts: each would
// read its operands from LDS for a quarter of the products.  The four multiplying wavefronts take the whole tile each
// and share out K instead -- a trip is 64 columns, four k-steps, one per wavefront -- and their sums meet in LDS at the
// end, added in wavefront order.  Per k-step a wavefront reads kFi + 2 kTj fragments for 2 kFi kTj MFMAs.
//
// The stages, the requesting wavefronts, the order of the pieces and the barrier are those of k_gemm_pipe; there are
// more and smaller stages, because what has to be in flight is weight bytes (4 KiB kFi a stage).
// kMode 2: the first half of the tile's rows are features of W1, the second half the same features of W3.
//
// What bounds it: the weights from HBM up to 64 tokens (W1+W3 of the 1B shape, 67 MB, 32 tokens: 49.6 us with the tile of
// 256 x 128 on 64 compute units, 15.4 here, of which launch, first data and epilogue are 4 to 5), the activations from L2
// into LDS beyond (128 tokens: 26 us, 268 MB in requests).  The workgroups of a die start their walk over K at different
// trips: in step, all of them would read the same columns of rows 4 KiB apart at once (W1+W3, 32 tokens: 19.4 -> 16.3 us).
// 32 prompt ids of the 1B shape: 1.90 -> 0.90 ms.
template <int kFi, int kTj, bool kLo>
struct FewShape {
    static constexpr int kRowBytes = 128;
    static constexpr int kRowsA = 32 * kFi, kRowsB = 32 * kTj, kRows = kRowsA + (kLo ? 2 : 1) * kRowsB;
    static constexpr int kStageBytes = kRows * kRowBytes;
    static constexpr int kLoads = kStageBytes / 4096;  // requests of 1 KiB per requesting wavefront and stage
    static constexpr int kStages = (160 * 1024) / kStageBytes > 10 ? 10 : (160 * 1024) / kStageBytes;
    static constexpr int kPitch = 36;  // floats per token row of a 32 x 32 tile of sums
    static constexpr int kSumBytes = 4 * kFi * kTj * 32 * kPitch * 4;
    static constexpr int kLdsBytes = kStages * kStageBytes > kSumBytes ? kStages * kStageBytes : kSumBytes;
    static_assert(kLdsBytes <= 160 * 1024 && kStages >= 3, "LDS of a workgroup");
};

template <int kFi, int kTj, int kMode, bool kLo, bool kRagged>
__global__ __launch_bounds__(512) void k_gemm_few(PipeJob job) {
    typedef FewShape<kFi, kTj, kLo> Shape;
    constexpr int kRowsA = Shape::kRowsA, kRowsB = Shape::kRowsB, kStages = Shape::kStages, kLoads = Shape::kLoads;
    constexpr int kStageBytes = Shape::kStageBytes, kRowBytes = Shape::kRowBytes, kPitch = Shape::kPitch;
    static_assert(kMode != 2 || kFi % 2 == 0, "as many tiles of W1 as of W3");
    extern __shared__ __align__(1024) char few_lds[];
    const int lane = lane_id();
    const int wave_of_8 = __builtin_amdgcn_readfirstlane(wave_index());
    const int wave = wave_of_8 & 3;
    const int id = static_cast<int>(blockIdx.x), die = id & 7, within = id >> 3;
    const int group = (within / job.token_tiles) * 8 + die;
    if (group >= job.groups) return;
    const int token_tile = within % job.token_tiles;
    const int tile_all = group % job.feature_tiles, split = group / job.feature_tiles;
    const int which = tile_all >= job.first_tile[2] ? 2 : (tile_all >= job.first_tile[1] ? 1 : 0);
    const int tile_x = tile_all - (which == 2 ? job.first_tile[2] : (which == 1 ? job.first_tile[1] : 0));
    const half_t* __restrict__ w = which == 2 ? job.w[2] : (which == 1 ? job.w[1] : job.w[0]);
    const int K = job.K, k_first = split * job.k_len, trips = job.k_len / 64;
    constexpr int kFeaturesPerTile = kMode == 2 ? 16 * kFi : 32 * kFi;
    const int f_base = tile_x * kFeaturesPerTile, t_base = token_tile * kRowsB;

    floatx16 acc[kFi][kTj];
    if (wave_of_8 >= 4) {
        const char* src[kLoads];
#pragma unroll
        for (int q = 0; q < kLoads; ++q) {
            const int row = 8 * (wave + 4 * q) + (lane >> 3);
            const int piece = (lane & 7) ^ ((row >> 1) & 7);
            const half_t* from;
            if (row < kRowsA) {
                if constexpr (kMode == 2) from = (row >= 16 * kFi ? job.w[1] : job.w[0]) + static_cast<size_t>(f_base + row % (16 * kFi)) * K;
                else from = w + static_cast<size_t>(f_base + row) * K;
            } else if (!kLo || row < kRowsA + kRowsB) {
                from = job.xh + static_cast<size_t>(t_base + row - kRowsA) * K;
            } else {
                from = job.xl + static_cast<size_t>(t_base + row - kRowsA - kRowsB) * K;
            }
            src[q] = reinterpret_cast<const char*>(from + k_first) + 16 * piece;
        }
        const unsigned lds_base = static_cast<unsigned>(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) char*)few_lds));
        const int turn0 = (group >> 3) % trips;
        // kRagged: of a wavefront's requests for token rows, eight rows each, those without a token are not made: its first
        // `made` of kTj for the heads, and as many for the remainders, are.  (What the rows hold then reaches their own columns
        // of the product only, and those are not stored.)
        auto request = [&](int trip, auto made) {
            const unsigned at = __builtin_amdgcn_readfirstlane(lds_base + (trip % kStages) * kStageBytes + wave * 1024);
            const int rot = trip + turn0 < trips ? trip + turn0 : trip + turn0 - trips;
            const int column = __builtin_amdgcn_readfirstlane(rot * kRowBytes);
#pragma unroll
            for (int q = 0; q < kLoads; ++q)
                if (q < kFi || (q - kFi) % kTj < made) {
                    const char* from = src[q] + column;
                    const unsigned to = at + q * 4096;
                    asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off\n" ::"v"(from), "s"(to) : "memory");
                }
        };
        auto landed = [&](int trip, auto made) {
            constexpr int kMade = kFi + (kLo ? 2 : 1) * decltype(made)::value;
            if (trips - 1 - trip >= kStages - 2) wait_requests<(kStages - 2) * kMade>();
            else wait_requests<0>();
        };
        auto feed = [&](auto made) {
#pragma unroll
            for (int t = 0; t < kStages - 1; ++t)
                if (t < trips) request(t, made);
            landed(0, made);
            __syncthreads();
            if (kStages - 1 < trips) request(kStages - 1, made);
            for (int t = 0; t < trips; ++t) {
                landed(t + 1, made);
                __syncthreads();
                if (t + kStages < trips) request(t + kStages, made);
            }
        };
        if constexpr (kRagged) {
            const int made = __builtin_amdgcn_readfirstlane(max(0, min(kTj, (job.live - t_base - 8 * wave + 31) / 32)));
            if (made >= kTj) feed(std::integral_constant<int, kTj>{});
            else if (kTj > 3 && made == 3) feed(std::integral_constant<int, kTj < 3 ? kTj : 3>{});
            else if (kTj > 2 && made == 2) feed(std::integral_constant<int, kTj < 2 ? kTj : 2>{});
            else if (kTj > 1 && made == 1) feed(std::integral_constant<int, 1>{});
            else feed(std::integral_constant<int, 0>{});
        } else {
            feed(std::integral_constant<int, kTj>{});
        }
    } else {
        const int r = lane & 31, g = lane >> 5;
        const int piece = (2 * wave + g) ^ ((r >> 1) & 7);  // this wavefront's k-step of every trip
        const int a_off = r * kRowBytes + 16 * piece, b_off = a_off + kRowsA * kRowBytes;
#pragma unroll
        for (int i = 0; i < kFi; ++i)
#pragma unroll
            for (int j = 0; j < kTj; ++j)
#pragma unroll
                for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.0f;
        struct Frags {
            half8_t a[kFi], bh[kTj], bl[kTj];
        };
        auto read = [&](Frags& f, int trip) {
            const char* stage = few_lds + (trip % kStages) * kStageBytes;
#pragma unroll
            for (int i = 0; i < kFi; ++i) f.a[i] = *reinterpret_cast<const half8_t*>(stage + a_off + i * 32 * kRowBytes);
#pragma unroll
            for (int j = 0; j < kTj; ++j) {
                f.bh[j] = *reinterpret_cast<const half8_t*>(stage + b_off + j * 32 * kRowBytes);
                if constexpr (kLo) f.bl[j] = *reinterpret_cast<const half8_t*>(stage + b_off + (kRowsB + j * 32) * kRowBytes);
            }
        };
        auto multiply = [&](const Frags& f) {
#pragma unroll
            for (int i = 0; i < kFi; ++i)
#pragma unroll
                for (int j = 0; j < kTj; ++j) {
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(f.a[i], f.bh[j], acc[i][j], 0, 0, 0);
                    if constexpr (kLo) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(f.a[i], f.bl[j], acc[i][j], 0, 0, 0);
                }
        };
        // (the trip's fragments are read behind the barrier that says they are there and multiplied behind the next
        // one: the reads travel while the trip before is multiplied.  The read past the last trip is of a stage nobody uses.)
        Frags even, odd;
        __syncthreads();
        read(even, 0);
        for (int t = 0; t < trips; t += 2) {
            __syncthreads();
            read(odd, t + 1);
            __builtin_amdgcn_sched_barrier(0);
            multiply(even);
            __builtin_amdgcn_sched_barrier(0);
            if (t + 1 < trips) {
                __syncthreads();
                read(even, t + 2);
                __builtin_amdgcn_sched_barrier(0);
                multiply(odd);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
    }
    // the four wavefronts' sums through LDS, tile by tile as [token][feature] (the stages are free: every wavefront has
    // read its last fragments, no request is outstanding), then whole lines to memory by all eight
    __syncthreads();
    float* sums = reinterpret_cast<float*>(few_lds);
    constexpr int kTile = 32 * kPitch;
    if (wave_of_8 < 4) {
        const int r = lane & 31, g = lane >> 5;
#pragma unroll
        for (int i = 0; i < kFi; ++i)
#pragma unroll
            for (int j = 0; j < kTj; ++j)
#pragma unroll
                for (int e4 = 0; e4 < 4; ++e4)
                    *reinterpret_cast<floatx4*>(sums + (wave * kFi * kTj + i * kTj + j) * kTile + r * kPitch + 8 * e4 + 4 * g) =
                        floatx4{acc[i][j][4 * e4], acc[i][j][4 * e4 + 1], acc[i][j][4 * e4 + 2], acc[i][j][4 * e4 + 3]};
    }
    __syncthreads();
    const int row8 = lane >> 3, part8 = lane & 7;
    auto summed = [&](int tile, int n) {
        floatx4 v[4];
#pragma unroll
        for (int z = 0; z < 4; ++z) v[z] = *reinterpret_cast<const floatx4*>(sums + (z * kFi * kTj + tile) * kTile + n * kPitch + 4 * part8);
        floatx4 sum;
#pragma unroll
        for (int e = 0; e < 4; ++e) sum[e] = (v[0][e] + v[1][e]) + (v[2][e] + v[3][e]);
        return sum;
    };
    // (a wavefront and turn: eight tokens of one tile)
    if constexpr (kMode == 2) {
        for (int turn = wave_of_8; turn < 2 * kFi * kTj; turn += 8) {
            const int tile = turn >> 2, i = tile / kTj, j = tile % kTj, n = 8 * (turn & 3) + row8;
            if (kRagged && t_base + 32 * j + n >= job.live) continue;
            const floatx4 g4 = summed(tile, n), u4 = summed(kFi / 2 * kTj + tile, n);
            const float gate[4] = {g4[0], g4[1], g4[2], g4[3]}, up[4] = {u4[0], u4[1], u4[2], u4[3]};
            half4_pf_t h, l;
            swiglu_split4(h, l, gate, up);
            const size_t at = static_cast<size_t>(t_base + 32 * j + n) * job.out_ld + f_base + 32 * i + 4 * part8;
            *reinterpret_cast<half4_pf_t*>(job.out_hi + at) = h;
            if constexpr (kLo) *reinterpret_cast<half4_pf_t*>(job.out_lo + at) = l;
        }
    } else {
        float* __restrict__ y = (which == 2 ? job.y[2] : (which == 1 ? job.y[1] : job.y[0])) + static_cast<size_t>(split) * job.split_stride;
        const int ldy = which == 2 ? job.ldy[2] : (which == 1 ? job.ldy[1] : job.ldy[0]);
        for (int turn = wave_of_8; turn < 4 * kFi * kTj; turn += 8) {
            const int tile = turn >> 2, i = tile / kTj, j = tile % kTj, n = 8 * (turn & 3) + row8;
            if (kRagged && t_base + 32 * j + n >= job.live) continue;
            floatx4 v = summed(tile, n);
            floatx4* out = reinterpret_cast<floatx4*>(y + static_cast<size_t>(t_base + 32 * j + n) * ldy + f_base + 32 * i + 4 * part8);
            if constexpr (kMode == 1) {
                const floatx4 old = *out;
                v = floatx4{old[0] + v[0], old[1] + v[1], old[2] + v[2], old[3] + v[3]};
            }
            *out = v;
        }
    }
}

// ---------------------------------------------------------------------------
// Causal attention over the cache
// ---------------------------------------------------------------------------
//
// One wavefront per (token t, KV head), four tokens to a workgroup: its query heads (gqa of
// them) attend to cache positions 0 .. pos0 + t (model.cpp:178-198; every row of the cache for these
// positions is in place, this chunk's included).  kGroup lanes share a position,
// 8 binary16 each; every lane group keeps a running maximum, sum and weighted V sum
// per query head (rescaled when the maximum grows), and the groups are merged by the
// same rule at the end.  Output: the heads' outputs, split into
// (hi, lo) for the output projection's GEMM.
// Sum over the kGroup lanes that share a position, by DPP moves (no LDS round trip).
template <int kGroup>
__device__ __forceinline__ float lanes_sum(float v) {
    static_assert(kGroup == 8 || kGroup == 16, "lane groups of 8 or 16");
    v += dpp_move<kDppXor1>(v);
    v += dpp_move<kDppXor2>(v);
    v += dpp_move<kDppHalfMirror>(v);
    if constexpr (kGroup == 16) v += dpp_move<kDppMirror>(v);
    return v;
}

// exp(x) as one hardware exponential (about an ulp off expf; the weights it forms are normalised
// by their own sum).
__device__ __forceinline__ float exp_fast(float x) { return __builtin_amdgcn_exp2f(x * 1.44269504088896341f); }

template <int kGroup>
__global__ __launch_bounds__(256) void k_attention(const float* __restrict__ q, const uint16_t* __restrict__ key_cache,
                                                   const uint16_t* __restrict__ value_cache, half_t* __restrict__ out_hi,
                                                   half_t* __restrict__ out_lo, int layer, int pos0, int dim, int kv_dim,
                                                   int hs, int gqa, int seq_len, int n_tokens) {
    constexpr int kGroups = kWave / kGroup;  // positions a wavefront covers per pass
    const int lane = lane_id(), wave = wave_index();
    const int t = static_cast<int>(blockIdx.x) * 4 + wave, kvh = blockIdx.y;
    if (t >= n_tokens) return;  // (wavefronts of a workgroup do not meet again)
    const int npos = pos0 + t + 1;
    const int sub = lane % kGroup, grp = lane / kGroup;
    const bool lane_live = sub * 8 < hs;
    const int off = lane_live ? sub * 8 : 0;
    const size_t head_base = static_cast<size_t>(layer) * kv_dim * seq_len + static_cast<size_t>(kvh) * seq_len * hs;
    const uint16_t* kbase = key_cache + head_base;
    const uint16_t* vbase = value_cache + head_base;
    const float scale = 1.0f / sqrtf(static_cast<float>(hs));  // model.cpp:188

    float qreg[kMaxGqa][8];
    float top[kMaxGqa], lsum[kMaxGqa], acc[kMaxGqa][8];
#pragma unroll
    for (int h = 0; h < kMaxGqa; ++h) {
        top[h] = -INFINITY;
        lsum[h] = 0.0f;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            acc[h][e] = 0.0f;
            qreg[h][e] = (h < gqa && lane_live) ? q[static_cast<size_t>(t) * dim + (kvh * gqa + h) * hs + off + e] : 0.0f;
        }
    }
    // (the rows of the position after this one are requested before this one's arithmetic; past the end
    // the last valid row is read again and dropped)
    const int first = grp;
    const int clamp = npos - 1;
    uintx4 k_next = load16(kbase + static_cast<size_t>(first < npos ? first : clamp) * hs + off);
    uintx4 v_next = load16(vbase + static_cast<size_t>(first < npos ? first : clamp) * hs + off);
    for (int p = first; p < npos; p += kGroups) {
        const half8_t kh = as_half8(k_next);
        const half8_t vh = as_half8(v_next);
        const int pn = p + kGroups;
        k_next = load16(kbase + static_cast<size_t>(pn < npos ? pn : clamp) * hs + off);
        v_next = load16(vbase + static_cast<size_t>(pn < npos ? pn : clamp) * hs + off);
#pragma unroll
        for (int h = 0; h < kMaxGqa; ++h) {
            if (h < gqa) {
                float s = 0.0f;
#pragma unroll
                for (int e = 0; e < 8; ++e) s = fmaf(static_cast<float>(kh[e]), qreg[h][e], s);
                s = lane_live ? s : 0.0f;
                s = lanes_sum<kGroup>(s) * scale;
                const float grown = fmaxf(top[h], s);
                const float corr = (top[h] == -INFINITY) ? 0.0f : exp_fast(top[h] - grown);
                const float pw = exp_fast(s - grown);
                top[h] = grown;
                lsum[h] = lsum[h] * corr + pw;
#pragma unroll
                for (int e = 0; e < 8; ++e) acc[h][e] = fmaf(static_cast<float>(vh[e]), pw, acc[h][e] * corr);
            }
        }
    }
    // lane groups of a wavefront
#pragma unroll
    for (int h = 0; h < kMaxGqa; ++h) {
        if (h < gqa) {
            float all = top[h];
#pragma unroll
            for (int o = kGroup; o < kWave; o <<= 1) all = fmaxf(all, __shfl_xor(all, o));
            const float f = (top[h] == -INFINITY) ? 0.0f : exp_fast(top[h] - all);
            float ls = lsum[h] * f;
#pragma unroll
            for (int o = kGroup; o < kWave; o <<= 1) ls += __shfl_xor(ls, o);
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                float v = acc[h][e] * f;
#pragma unroll
                for (int o = kGroup; o < kWave; o <<= 1) v += __shfl_xor(v, o);
                acc[h][e] = v;
            }
            if (grp == 0 && lane_live) {
#pragma unroll
                for (int e = 0; e < 8; ++e)
                    split_store(out_hi, out_lo, static_cast<size_t>(t) * dim + (kvh * gqa + h) * hs + off + e, acc[h][e] / ls);
            }
        }
    }
}

// ---------------------------------------------------------------------------
// The same attention on the matrix cores
// ---------------------------------------------------------------------------
//
// A wavefront owns 32 query rows = (32 / gqa) consecutive tokens x the gqa query heads of one KV head, and walks the
// context in steps of 32 positions.  A workgroup is kR x kP such wavefronts: kR take neighbouring rows and share every
// step's K and V rows, kP take the steps in turn and merge their running (maximum, sum, output) at the end.  2 x 2 where
// that makes workgroups enough; a batch of few rows takes 1 x 8 or 1 x 4 (heads of 128: 1 x 4, for want of LDS).  Per step:
//   S^T[pos][row] = sum_d K[pos][d] Q[row][d]     A = K rows, B = Q (head + remainder, in registers for the whole walk)
//   online softmax: in the result a LANE holds one query row (its column) and 16 of the 32 positions, the lane 32 further
//                   on the other 16 -- maximum and rescaling are per lane, with one exchange between the two halves of
//                   the wavefront per step; the sums of the two halves meet once, at the end
//   O^T[d][row] += sum_pos V^T[d][pos] P^T[pos][row]   A = V transposed, B = P straight from the lane's own registers
// A lane's 16 positions of 32 are {8j + 4g .. 8j + 4g + 3 : j = 0..3} (g = lane / 32), so as B operand of the second
// product it supplies, per 16 positions, positions 4g..4g+3 and 8+4g..8+4g+3; V is read in the same order (any
// permutation of k is fine as long as both operands use it).  Queries and probabilities are split into binary16 head +
// remainder like every other activation.  The softmax works in powers of two; log2(e) / sqrt(head size) goes into the fp32
// score, in the one fma that takes the reference off it: multiplied into the queries, it would take five sixths off them
// before the split, and the remainders of queries below about 0.7 would lose bits to binary16's subnormals.
//
// K and V rows travel from the cache into LDS by requests of 1 KiB (no registers, and nothing waits but the step that
// reads them), a step ahead.  The 16-byte pieces of a row are stored in an order that keeps the reads free of bank
// conflicts (the address each lane requests makes it): K fragments are 16 bytes a lane from 32 rows; V fragments are
// transposed on the way out (ds_read_b64_tr_b16: 16 lanes read a tile of 4 positions x 16 dimensions and every lane gets
// the 4 positions of one dimension).  Rows past the workgroup's last position are the last row again.
//
// A weight of zero does not keep an infinite value out of the output, so a wavefront must not multiply the V rows of its
// neighbour's positions.  It has them in one step, the one its own last position ends in, and takes that step's V rows
// from a copy in LDS with the neighbour's rows cleared.  (Cleared in the fragments, behind a branch in every step or by
// masks, the registers and clocks cost every step: 1B shape, 2000 ids behind 3000, 10.28 -> 10.47 and 10.57 ms exact,
// 6.93 -> 7.11 and 7.29 fast; with the copy 10.06 -> 10.05 and 6.86 -> 6.93.)
//
// What bounds it: a step of 32 positions is 512 MFMA clocks and about as many of the vector units (sixteen v_exp_f32 are
// 256 of them), and one wavefront does them one after the other, so what counts is wavefronts per SIMD: the stages are
// kept small enough for two to four workgroups to a compute unit.  (Measured and not better: the next step's scores
// formed between this step's weights in the same wavefront, at twice the stages; more steps in flight; 128 rows to a
// workgroup; a short batch's context split over several workgroups with a kernel that merges them.)  1B shape, exact
// mode: 150 ids behind 3000, 34 -> 22 us a layer; 2048 ids behind 2048, 107 us on average.

typedef _Float16 half4_t __attribute__((ext_vector_type(4)));
typedef _Float16 half2_t __attribute__((ext_vector_type(2)));
typedef short short4_t __attribute__((ext_vector_type(4)));

template <int kHs, int kR, int kP>
struct AttentionShape {
    static constexpr int kStep = 32;
    static constexpr int kRowBytes = 2 * kHs, kPieces = kHs / 8;
    static constexpr int kHalfBytes = kStep * kRowBytes, kStageBytes = 2 * kHalfBytes;  // K rows, then V rows
    static constexpr int kLoads = kStageBytes / 1024 / kR;                              // requests per wavefront and step
    // 2 x 2: 36 / 72 KiB, four or two workgroups to a compute unit (heads of 64 in three stages, 52 KiB: three of them, and
    // of 2048 ids' 1024 workgroups a last round with one wavefront to a SIMD; behind 2048 positions 119.5 us, 111.1 so)
    static constexpr int kStages = 2;
    static constexpr int kPartFloats = (kHs / 2 + 2) * 64;  // a wavefront's maximum, sum and output
    static constexpr int kMergeBytes = kP * kR * kPartFloats * 4;
    static_assert(kP > 1 && kHs / 8 % kP == 0, "the output's pieces are shared out among the wavefronts of a row");
    // behind the stages: V rows of a step, for each row of wavefronts but the last
    static constexpr int kOwnValues = kP * kStages * kStageBytes;
    static constexpr int kStepBytes = kOwnValues + (kR - 1) * kHalfBytes;
    static constexpr int kLdsBytes = kStepBytes > kMergeBytes ? kStepBytes : kMergeBytes;
    static_assert(kLdsBytes <= 160 * 1024, "LDS of a workgroup");
};

// max(v, the other half-wavefront's v) / v + the other half-wavefront's v
__device__ __forceinline__ float halves_max(float v) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float halves_sum(float v) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// (p0, p1) rounded to binary16, and what is left of each (exact).  The packed pair and the factor -1 are hidden from the
// compiler, which would otherwise round every value a second time to subtract it: one v_cvt_pk_f16_f32 and two v_fma_mix_f32.
// (No instruction is written here by hand: one that reads a result of v_exp_f32 needs a wait state, which the compiler
// counts for its own instructions only.)
__device__ __forceinline__ half2_t split_pair(float& p0, float& p1, float minus_one) {
    uint32_t packed = __builtin_bit_cast(uint32_t, half2_t{static_cast<half_t>(p0), static_cast<half_t>(p1)});
    asm("" : "+v"(packed));
    const half2_t h = __builtin_bit_cast(half2_t, packed);
    p0 = fmaf(static_cast<float>(h[0]), minus_one, p0);
    p1 = fmaf(static_cast<float>(h[1]), minus_one, p1);
    return h;
}

template <int kHs, bool kLo, int kR, int kP>
__global__ __launch_bounds__(64 * kR * kP, 2) void k_attention_mfma(const float* __restrict__ q, const uint16_t* __restrict__ key_cache,
                                                                 const uint16_t* __restrict__ value_cache,
                                                                 half_t* __restrict__ out_hi, half_t* __restrict__ out_lo, int layer,
                                                                 int pos0, int dim, int kv_dim, int gqa, int seq_len, int n_tokens,
                                                                 int round_tiles) {
    typedef AttentionShape<kHs, kR, kP> Shape;
    constexpr int kDTiles = kHs / 32, kKSteps = kHs / 16, kStep = Shape::kStep, kRowBytes = Shape::kRowBytes;
    constexpr int kPieces = Shape::kPieces, kLoads = Shape::kLoads, kHalfBytes = Shape::kHalfBytes, kStageBytes = Shape::kStageBytes;
    constexpr int kStages = Shape::kStages;
    extern __shared__ __align__(1024) char att_lds[];
    const int lane = lane_id();
    const int wave = __builtin_amdgcn_readfirstlane(wave_index());
    const int wr = wave % kR, wp = wave / kR;
    const int r = lane & 31, g = lane >> 5;
    const int tokens_per_wave = 32 / gqa;
    // (one KV head after the other in the workgroup's number: where there are as many KV heads as dies, a head's rows
    // stay in one die's L2.  The tiles with the longest contexts are dispatched first; where the device takes two rounds of
    // workgroups at once, the second round's go out shortest first, so that a compute unit has a long and a short one.)
    const int kvh = blockIdx.x, round = round_tiles > 0 ? static_cast<int>(blockIdx.y) / round_tiles : 0;
    const int first_of_round = round * round_tiles, after_round = min(first_of_round + round_tiles, static_cast<int>(gridDim.y));
    const int order = (round & 1) ? after_round - 1 - (static_cast<int>(blockIdx.y) - first_of_round) : static_cast<int>(blockIdx.y);
    const int tile = static_cast<int>(gridDim.y) - 1 - order;
    const int first_token = tile * kR * tokens_per_wave;                                         // of the workgroup
    const int t0 = first_token + wr * tokens_per_wave;                                           // of the wavefront
    // positions below which `token`s before attend
    auto end_of = [&](int token) { return pos0 + (token < n_tokens ? token : n_tokens); };
    const int limit = end_of(first_token + kR * tokens_per_wave);                // the workgroup reads [0, limit)
    const int wave_limit = t0 < n_tokens ? end_of(t0 + tokens_per_wave) : 0;     // the wavefront attends to [0, wave_limit)
    const int my_tok = t0 + r / gqa, my_head = r % gqa;
    const bool valid = my_tok < n_tokens;
    const int tok_c = valid ? my_tok : n_tokens - 1;
    const int my_limit = pos0 + tok_c + 1;                                       // this lane's row attends to [0, my_limit)
    const size_t head_base = static_cast<size_t>(layer) * kv_dim * seq_len + static_cast<size_t>(kvh) * seq_len * kHs;
    const char* kbase = reinterpret_cast<const char*>(key_cache + head_base);
    const char* vbase = reinterpret_cast<const char*>(value_cache + head_base);

    char* stages = att_lds + wp * kStages * kStageBytes;
    const unsigned lds_base = static_cast<unsigned>(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) char*)stages));
    const int steps = (limit + kStep - 1) / kStep, turns = (steps + kP - 1) / kP;
    constexpr int kRowsPerLoad = 1024 / kRowBytes, kLoadsPerHalf = kHalfBytes / 1024;
    auto request = [&](int turn) {
        const int p0 = (turn * kP + wp) * kStep;
#pragma unroll
        for (int i = 0; i < kLoads; ++i) {
            const int load = wr + kR * i, in_half = load % kLoadsPerHalf;
            const bool is_v = load >= kLoadsPerHalf;  // (uniform)
            const int row = in_half * kRowsPerLoad + lane / kPieces;
            const int swizzle = is_v ? (kHs == 64 ? 4 * ((row >> 1) & 1) : 4 * (row & 3)) : (kHs == 64 ? (row >> 1) & 7 : row & 15);
            const int pos = p0 + row < limit ? p0 + row : limit - 1;
            const char* src = (is_v ? vbase : kbase) + static_cast<size_t>(pos) * kRowBytes + 16 * ((lane % kPieces) ^ swizzle);
            const unsigned at = __builtin_amdgcn_readfirstlane(lds_base + (turn % kStages) * kStageBytes + load * 1024);
            asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off\n" ::"v"(src), "s"(at) : "memory");
        }
    };
#pragma unroll
    for (int t = 0; t < kStages - 1; ++t)
        if (t < turns) request(t);

    half8_t qh[kKSteps], ql[kKSteps];
    {
        const float* qrow = q + static_cast<size_t>(tok_c) * dim + (kvh * gqa + my_head) * kHs + 8 * g;
#pragma unroll
        for (int s = 0; s < kKSteps; ++s)
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const float v = qrow[16 * s + e];
                const half_t h = static_cast<half_t>(v);
                qh[s][e] = h;
                ql[s][e] = static_cast<half_t>(v - static_cast<float>(h));
            }
    }
    floatx16 o[kDTiles];
#pragma unroll
    for (int dt = 0; dt < kDTiles; ++dt)
#pragma unroll
        for (int e = 0; e < 16; ++e) o[dt][e] = 0.0f;
    // Weights are 2^(scale * score - top).  The reference `top` follows the row's maximum lazily: it moves only when a
    // step's maximum exceeds it by more than kSlack (weights then stay below 2^kSlack, far inside binary16, and any reference
    // gives the same quotient in the end).  After a row's first steps it hardly ever moves, and a step in which no row's
    // reference moved rescales nothing.  In the exact mode it is a whole number, so that rescaling and merging multiply by
    // powers of two and round nothing (in the fast mode the largest weight, if it is 1, is the one that binary16 holds exactly).
    // The products start from zero: from -top, every partial sum would be rounded at the size of the row's maximum.
    // 8B shape, 140 ids, the cache of all layers against float64: 3.50e-4 with scaled queries and products from -top, 3.40e-4
    // so.
    constexpr float kSlack = 6.0f;
    const float scale = 1.44269504088896341f / sqrtf(static_cast<float>(kHs));  // model.cpp:188
    float top = 0.0f, lsum = 0.0f;  // (the sum over this lane's own positions)
    bool seen = false;              // the row has attended to something: top is a score
    float minus_one = -1.0f;
    asm("" : "+v"(minus_one));

    // where this lane reads its fragments of a step: K row r, pieces 2 s + g; V rows 4 g + (lane % 16) / 4 of the first
    // sixteen, dimensions 32 dt + 16 (lane / 16 % 2) + 4 (lane % 4) ..
    int k_at[kKSteps], v_at[kDTiles];
#pragma unroll
    for (int s = 0; s < kKSteps; ++s) k_at[s] = r * kRowBytes + 16 * ((2 * s + g) ^ (kHs == 64 ? (r >> 1) & 7 : r & 15));
    {
        const int row = 4 * g + ((lane & 15) >> 2);
#pragma unroll
        for (int dt = 0; dt < kDTiles; ++dt) {
            const int piece = 4 * dt + 2 * ((lane >> 4) & 1) + ((lane & 3) >> 1);
            v_at[dt] = row * kRowBytes + 16 * (piece ^ (kHs == 64 ? 4 * ((row >> 1) & 1) : 4 * (row & 3))) + 8 * (lane & 1);
        }
    }

    for (int turn = 0; turn < turns; ++turn) {
        const int p0 = (turn * kP + wp) * kStep;
        // (the step's rows have landed, and nobody reads the stage the next requests go to any more)
        if (turns - 1 - turn >= kStages - 2) wait_requests<(kStages - 2) * kLoads>();
        else wait_requests<0>();
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        if constexpr (kR > 1) __syncthreads();
        if (turn + kStages - 1 < turns) request(turn + kStages - 1);
        if (p0 >= wave_limit) continue;
        const char* stage = stages + (turn % kStages) * kStageBytes;
        const char* values = stage + kHalfBytes;
        if constexpr (kR > 1) {
            if (p0 + kStep > wave_limit && wave_limit < limit) {  // (uniform; one wavefront of its row, one step)
                char* own = att_lds + Shape::kOwnValues + wr * kHalfBytes;
#pragma unroll
                for (int i = 0; i < kLoadsPerHalf; ++i) {
                    uintx4 v = *reinterpret_cast<const uintx4*>(values + 1024 * i + 16 * lane);
                    if (p0 + i * kRowsPerLoad + lane / kPieces >= wave_limit) v = uintx4{0u, 0u, 0u, 0u};
                    *reinterpret_cast<uintx4*>(own + 1024 * i + 16 * lane) = v;
                }
                values = own;
            }
        }
        floatx16 st;
#pragma unroll
        for (int e = 0; e < 16; ++e) st[e] = 0.0f;
#pragma unroll
        for (int s = 0; s < kKSteps; ++s) {
            const half8_t kf = *reinterpret_cast<const half8_t*>(stage + k_at[s]);
            st = __builtin_amdgcn_mfma_f32_32x32x16_f16(kf, qh[s], st, 0, 0, 0);
            if constexpr (kLo) st = __builtin_amdgcn_mfma_f32_32x32x16_f16(kf, ql[s], st, 0, 0, 0);
        }
        if (p0 + kStep > pos0 + t0 + 1) {  // (uniform) some row of the wavefront does not attend to the whole step
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                const int pos = p0 + 8 * (e >> 2) + 4 * g + (e & 3);
                st[e] = pos < my_limit ? st[e] : -INFINITY;
            }
        }
        float step_top = -INFINITY;
#pragma unroll
        for (int e = 0; e < 16; ++e) step_top = fmaxf(step_top, st[e]);
        step_top = halves_max(step_top) * scale;
        if constexpr (kLo) step_top = __builtin_ceilf(step_top);
        const bool moves = step_top > (seen ? top + kSlack : -INFINITY);
        if (__builtin_amdgcn_ballot_w64(moves) != 0ull) {  // (uniform)
            const float to = moves ? step_top : top;
            const float corr = __builtin_amdgcn_exp2f(seen ? top - to : 0.0f);  // (nothing to rescale before a row's first step)
            top = to;
            lsum *= corr;
#pragma unroll
            for (int dt = 0; dt < kDTiles; ++dt)
#pragma unroll
                for (int e = 0; e < 16; ++e) o[dt][e] *= corr;
            seen = seen || moves;
        }
        float step_sum = 0.0f;  // (of its own, so that the running sum is rounded once a step)
#pragma unroll
        for (int s2 = 0; s2 < 2; ++s2) {
            half8_t ph, pl;
#pragma unroll
            for (int e = 0; e < 8; e += 2) {
                float p_0 = __builtin_amdgcn_exp2f(fmaf(st[8 * s2 + e], scale, -top)), p_1 = __builtin_amdgcn_exp2f(fmaf(st[8 * s2 + e + 1], scale, -top));
                step_sum += p_0 + p_1;
                half2_t h;
                if constexpr (kLo) h = split_pair(p_0, p_1, minus_one);
                else h = half2_t{static_cast<half_t>(p_0), static_cast<half_t>(p_1)};
                ph[e] = h[0];
                ph[e + 1] = h[1];
                if constexpr (kLo) {
                    pl[e] = static_cast<half_t>(p_0);
                    pl[e + 1] = static_cast<half_t>(p_1);
                }
            }
#pragma unroll
            for (int dt = 0; dt < kDTiles; ++dt) {
                union {
                    short4_t part[2];
                    half8_t whole;
                } vf;
#pragma unroll
                for (int j = 0; j < 2; ++j)
                    vf.part[j] = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                        (__attribute__((address_space(3))) short4_t*)(values + v_at[dt] + (16 * s2 + 8 * j) * kRowBytes));
                o[dt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vf.whole, ph, o[dt], 0, 0, 0);
                if constexpr (kLo) o[dt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vf.whole, pl, o[dt], 0, 0, 0);
            }
        }
        lsum += step_sum;
    }
    lsum = halves_sum(lsum);
    if (!seen) top = -INFINITY;
    // The wavefronts of a row meet in LDS, lane for lane: each leaves its (maximum, sum, output), and each adds up its share of
    // the output's pieces of four values in the order of the wavefronts (one wavefront for all of them, the others gone:
    // 1B shape, 32 ids: 7.2 us a launch, 6.15 this way; 8B, 150 ids: 9.8 and 9.2).  Those past the context's last step have
    // left nothing and are not read.
    // Of the first two parts one is rounded with its weight on its own and the other added by a fused multiply-add.  Which one
    // is written out and stays as it is, the second part for the sums and the outputs of heads of 64, the first for the
    // outputs of heads of 128: the weights of the fast mode are no powers of two, and the other choice moves last bits of
    // outputs, which the binary16 inputs of the products behind them turn into 8e-4 of the cache (1B shape, 2011 ids).
    __syncthreads();  // (the stages are free)
    constexpr int kFours = kHs / 8, kPart = Shape::kPartFloats;  // pieces of four values, floats of a wavefront's part
    const int parts = steps < kP ? steps : kP;
    float* merge = reinterpret_cast<float*>(att_lds) + wr * kP * kPart;
    if (wp < parts) {
        float* mine = merge + wp * kPart;
        mine[lane] = top;
        mine[64 + lane] = lsum;
#pragma unroll
        for (int four = 0; four < kFours; ++four)
            *reinterpret_cast<floatx4*>(mine + 128 + 256 * four + 4 * lane) =
                floatx4{o[four >> 2][4 * (four & 3)], o[four >> 2][4 * (four & 3) + 1], o[four >> 2][4 * (four & 3) + 2], o[four >> 2][4 * (four & 3) + 3]};
    }
    __syncthreads();
    float weight[kP], all_top = -INFINITY, total;
#pragma unroll
    for (int w = 0; w < kP; ++w) {
        weight[w] = w < parts ? merge[w * kPart + lane] : -INFINITY;
        all_top = fmaxf(all_top, weight[w]);
    }
    if (all_top == -INFINITY) all_top = 0.0f;  // (a row past the last token)
#pragma unroll
    for (int w = 0; w < kP; ++w) weight[w] = __builtin_amdgcn_exp2f(weight[w] - all_top);
    auto sum_of = [&](int w) { return w < parts ? merge[w * kPart + 64 + lane] : 0.0f; };
    total = fmaf(sum_of(0), weight[0], sum_of(1) * weight[1]);
#pragma unroll
    for (int w = 2; w < kP; ++w) total = fmaf(sum_of(w), weight[w], total);
    if (!valid) return;
    const size_t base = static_cast<size_t>(my_tok) * dim + (kvh * gqa + my_head) * kHs;
    const float inv_sum = 1.0f / total;
#pragma unroll
    for (int f = 0; f < kFours / kP; ++f) {
        const int four = wp + kP * f;
        auto part_of = [&](int w) { return *reinterpret_cast<const floatx4*>(merge + w * kPart + 128 + 256 * four + 4 * lane); };
        const floatx4 first = part_of(0), second = parts > 1 ? part_of(1) : floatx4{0.0f, 0.0f, 0.0f, 0.0f};
        floatx4 v;
#pragma unroll
        for (int u = 0; u < 4; ++u)
            v[u] = kHs == 64 ? fmaf(first[u], weight[0], second[u] * weight[1]) : fmaf(second[u], weight[1], first[u] * weight[0]);
#pragma unroll
        for (int w = 2; w < kP; ++w) {
            if (w >= parts) break;
            const floatx4 a = part_of(w);
#pragma unroll
            for (int u = 0; u < 4; ++u) v[u] = fmaf(a[u], weight[w], v[u]);
        }
        half4_t h, l;
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            v[u] *= inv_sum;
            h[u] = static_cast<half_t>(v[u]);
            l[u] = static_cast<half_t>(v[u] - static_cast<float>(h[u]));
        }
        const size_t at = base + 32 * (four >> 2) + 8 * (four & 3) + 4 * g;
        *reinterpret_cast<half4_t*>(out_hi + at) = h;
        if constexpr (kLo) *reinterpret_cast<half4_t*>(out_lo + at) = l;
    }
}

// x[i] (+)= p[0][i] + p[1][i] + ... in that order: the partial products of a GEMM whose K was split.
template <bool kAccumulate>
__global__ __launch_bounds__(256) void k_add_partials(float* __restrict__ x, const float* __restrict__ p, int splits,
                                                      size_t stride, size_t count) {
    const size_t i = (static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x) * 4;
    if (i >= count) return;
    floatx4 v = kAccumulate ? *reinterpret_cast<const floatx4*>(x + i) : floatx4{0.0f, 0.0f, 0.0f, 0.0f};
    for (int s = 0; s < splits; ++s) {
        const floatx4 a = *reinterpret_cast<const floatx4*>(p + s * stride + i);
        v = floatx4{v[0] + a[0], v[1] + a[1], v[2] + a[2], v[3] + a[3]};
    }
    *reinterpret_cast<floatx4*>(x + i) = v;
}

// (hi, lo) = x as it is (the GEMM entry point's own inputs).
__global__ __launch_bounds__(256) void k_split(const float* __restrict__ x, half_t* __restrict__ hi, half_t* __restrict__ lo,
                                               size_t count) {
    const size_t i = static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i < count) split_store(hi, lo, i, x[i]);
}

}  // namespace pf

// ---------------------------------------------------------------------------
// Host side
// ---------------------------------------------------------------------------

namespace {

// Buffers of a chunk of t_pad tokens, in lpp_model::pf_buf order: parts of one allocation, which kBufAll names.
enum { kBufTokens, kBufX, kBufQ, kBufK, kBufV, kBufPartials, kBufHi, kBufLo, kBufHi2, kBufLo2, kBufAll, kBufCount };
static_assert(kBufCount <= static_cast<int>(sizeof(lpp_model::pf_buf) / sizeof(void*)), "lpp_model::pf_buf is too small");

const char* unsupported_reason(const lpp_model* m) {
    const lpp_config& c = m->cfg;
    if (c.weight_precision != LPP_WEIGHT_FP16) return "weights are not binary16";
    if (c.dim % pf::kTileFeatures != 0 || m->kv_dim % pf::kTileFeatures != 0 || c.hidden_dim % pf::kTileFeatures != 0)
        return "dim, kv_dim and hidden_dim must be multiples of 128";
    if (m->head_size != 64 && m->head_size != 128) return "head_size must be 64 or 128";
    if (m->gqa > pf::kMaxGqa) return "more than 8 query heads per KV head";
    return nullptr;
}

// Y_i[t][f] (+)= sum_k W_i[f][k] * x[t][k] for up to three matrices W_i of n_i rows that share x.
struct Product {
    const void* w;
    float* y;
    int n;
};

// A kernel's LDS need, told to the runtime once per device (the attribute belongs to the device's copy of the kernel).
lpp_status size_lds(const void* kernel, int bytes, bool (&sized)[64]) {
    int device = 0;
    LPP_HIP(hipGetDevice(&device));
    if (device < 0 || device >= 64 || !sized[device]) {
        LPP_HIP(hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, bytes));
        if (device >= 0 && device < 64) sized[device] = true;
    }
    return LPP_OK;
}
template <int kFi, int kTj, int kMode, bool kLo = true, bool kRagged = false>
lpp_status size_pipe() {
    static bool sized[64] = {};
    return size_lds(reinterpret_cast<const void*>(&pf::k_gemm_pipe<kFi, kTj, kMode, kLo, kRagged>),
                    pf::PipeShape<kFi, kTj, kLo>::kLdsBytes, sized);
}
template <int kFi, int kTj, int kMode, bool kLo, bool kRagged = false>
lpp_status size_few() {
    static bool sized[64] = {};
    return size_lds(reinterpret_cast<const void*>(&pf::k_gemm_few<kFi, kTj, kMode, kLo, kRagged>), pf::FewShape<kFi, kTj, kLo>::kLdsBytes, sized);
}

template <int kFi, int kTj, int kMode, bool kLo, bool kRagged>
lpp_status launch_pipe_as(const pf::PipeJob& job, hipStream_t s) {
    typedef pf::PipeShape<kFi, kTj, kLo> Shape;
    LPP_TRY((size_pipe<kFi, kTj, kMode, kLo, kRagged>()));
    const int per_die = (job.groups + 7) / 8;
    hipLaunchKernelGGL((pf::k_gemm_pipe<kFi, kTj, kMode, kLo, kRagged>), dim3(per_die * 8 * job.token_tiles), dim3(512), Shape::kLdsBytes, s,
                       job);
    LPP_CHECK_LAUNCH("k_gemm_pipe");
    return LPP_OK;
}
// (a job without a remainder array takes the kernels that neither fetch nor multiply one)
//
// Tokens are padded to 128.  In the exact mode the device's power is what limits the products of a full tile, and columns of
// 32 that hold no token take as much of it: where they are a twelfth of all or more, the kernels that leave them out are
// the faster ones (1B shape, 300 ids, 2 of 12: 2.14 -> 2.06 ms, 200, 1 of 8: 1.68 -> 1.66; of 450 ids, 1 of 16, 2.472 ->
// 2.495).  The tokens are dealt out evenly where that makes every tile narrower: 150 ids as 96 + 54, 1.585 -> 1.495 ms; 8B
// shape 7.73 -> 7.05.  In the fast mode only that pays: 150 ids 1.417 -> 1.280, 257 ids 1.721 -> 1.625, but 200 ids, cut
// 128 + 72 either way, 1.454 -> 1.463.
template <int kFi, int kTj, int kMode>
lpp_status launch_pipe(const pf::PipeJob& job_in, hipStream_t s) {
    pf::PipeJob job = job_in;
    const int columns = (job.live + 31) / 32, all = 2 * kTj * job.token_tiles;
    job.each = 32 * ((columns + job.token_tiles - 1) / job.token_tiles);
    if (job.xl != nullptr ? 12 * (all - columns) >= all : job.each < 64 * kTj)
        return job.xl != nullptr ? launch_pipe_as<kFi, kTj, kMode, true, true>(job, s)
                                 : launch_pipe_as<kFi, kTj, kMode, false, true>(job, s);
    return job.xl != nullptr ? launch_pipe_as<kFi, kTj, kMode, true, false>(job, s)
                             : launch_pipe_as<kFi, kTj, kMode, false, false>(job, s);
}

template <int kMode, bool kLo>
lpp_status size_block() {
    static bool sized[64] = {};
    return size_lds(reinterpret_cast<const void*>(&pf::k_gemm_block<kMode, kLo>), pf::BlockShape<kLo>::kLdsBytes, sized);
}
template <int kMode, bool kLo>
lpp_status launch_block(pf::PipeJob job, hipStream_t s) {
    LPP_TRY((size_block<kMode, kLo>()));
    job.band = job.token_tiles;
    hipLaunchKernelGGL((pf::k_gemm_block<kMode, kLo>), dim3((job.groups + 7) / 8 * 8 * job.token_tiles), dim3(512), pf::BlockShape<kLo>::kLdsBytes, s, job);
    LPP_CHECK_LAUNCH("k_gemm_block");
    return LPP_OK;
}

template <int kFi, int kTj, int kMode, bool kLo, bool kRagged>
lpp_status launch_few_as(const pf::PipeJob& job, hipStream_t s) {
    constexpr int kLds = pf::FewShape<kFi, kTj, kLo>::kLdsBytes;
    LPP_TRY((size_few<kFi, kTj, kMode, kLo, kRagged>()));
    const int per_die = (job.groups + 7) / 8;
    hipLaunchKernelGGL((pf::k_gemm_few<kFi, kTj, kMode, kLo, kRagged>), dim3(per_die * 8 * job.token_tiles), dim3(512), kLds, s, job);
    LPP_CHECK_LAUNCH("k_gemm_few");
    return LPP_OK;
}
// kRagged where at least eight of the last tile's rows are no token's.  A full tile through it takes 0.4 us a launch longer (128
// ids of the TinyLlama shape 1.69 -> 1.73 ms: the kernel has a loop for every number of requests, and starts with cold
// instructions), so it has its own; exact mode, before and with it: TinyLlama 10 ids 1.16 -> 1.06 ms, 22 1.16 -> 1.10, 72
// 1.50 -> 1.42; 1B 24 ids 0.92 -> 0.87; 8B 10 ids 4.18 -> 3.60, 40 4.67 -> 4.19.
template <int kFi, int kTj, int kMode, bool kLo>
lpp_status launch_few(const pf::PipeJob& job, hipStream_t s) {
    const bool ragged = job.live <= 32 * kTj * job.token_tiles - 8;
    return ragged ? launch_few_as<kFi, kTj, kMode, kLo, true>(job, s) : launch_few_as<kFi, kTj, kMode, kLo, false>(job, s);
}

// How a product is laid out on the device: what a workgroup's tile is and in how many ranges K is cut.
struct Plan {
    bool few;          // k_gemm_few (rows = 32 fi, tokens = 32 tj), otherwise k_gemm_pipe (rows = 64 fi, tokens = 64 tj)
    int fi, tj;        // ({false, 4, 4}: k_gemm_block)
    int splits;
    bool block() const { return !few && tj == 4; }
    int tile_rows() const { return (few ? 32 : 64) * fi; }
    int tile_tokens() const { return (few ? 32 : 64) * tj; }
    // Tiles of k_gemm_few that hold a token (150 ids, Wo in tiles of 64: three of four; 1B shape 1.466 -> 1.455 ms);
    // k_gemm_pipe deals the tokens out (launch_pipe).  Beyond 128 tokens the plan itself goes by t_pad: by the tokens it would
    // take Wo of 130 to 160 ids for k_gemm_pipe's tile of 96, 1.5 % faster there and 2.4 % slower at 192.
    int token_tiles(int t_pad, int live) const { return ((few ? live : t_pad) + tile_tokens() - 1) / tile_tokens(); }
};

// Rows the activations of n tokens are padded to: whole tiles of 128 tokens, or of 32 up to 64 (up to 96, k_gemm_pipe, whose
// tiles need rows of 128, was out of reach of 65 to 96 ids: 8B shape, 96 ids 5.75 ms, 128 ids 5.25).
int padded_tokens(int n) {
    const int unit = n <= 64 && test_option(LPP_OPT_PREFILL_STAGED_GEMM) != 0 ? 32 : pf::kTileTokens;
    return (n + unit - 1) / unit * unit;
}

// More than 256 tokens: k_gemm_pipe's tiles of 128 or 256 rows or k_gemm_block, K in one range or several, by the rounds of
// workgroups a launch of each makes.  A larger tile has fewer bytes to a product, a smaller one, or more ranges, fills the
// device better.  A round costs a launch's share that does not depend on K, and K columns; a last round of a few workgroups
// costs two thirds of a full one or more, and no launch less than one; partial products are written and read at 2.8 TB/s.
// The constants are a fit to 4100 timed prefills (TinyLlama, 1B and 8B shapes, 300 to 2036 ids, both modes, each tile and cut
// for each of the four products in turn; a column of 256 x 128, and that tile's last round in the fast mode, adjusted since to
// its trips of 64 columns).  By the fit a prefill was within 1 % of what that product's fastest launch makes it, and it is
// faster than by rules that cut K only while all ranges fit the device at once: exact mode, 8B shape 370 ids 11.9 -> 10.7 ms,
// 600 18.6 -> 17.1, 750 20.4 -> 19.6; 1B 1140 5.21 -> 4.91; TinyLlama 1530 7.53 -> 7.17.
// W1+W3, tiles against blocks: 1B shape 1024 ids 127 / 81 and 118 / 67 us, 1280 ids (a quarter of a second round) 163 / 108
// and 187 / 113, 2048 ids 236 / 156 and 217 / 127; 8B 512 ids 224 / 152 and 196 / 122, 1024 ids 426 / 280 and 369 / 224.
//
// Up to 256 tokens the choice is made by what a launch of each would take.  A workgroup is paced by its bytes from L2 into
// LDS, one of k_gemm_pipe, in the exact mode up to 128 tokens, by its MFMA clocks where they take longer; a last round of
// workgroups that does not fill the device counts almost whole; k_gemm_few's sums meet in LDS, a tile of 32 x 32 at a time;
// every partial product of a cut K is written, in many short runs, and read once more.  No launch is faster than
// its weights, and of two that are bound by them the one with less to do is taken.  The constants are a fit to 10000 timed
// prefills (TinyLlama, 1B and 8B shapes, 10 to 256 ids, both modes, every tile of the list for each of the four products in
// turn): up to 128 tokens a prefill is 0.3 % slower on average than with that product's fastest launch.  In the exact mode
// beyond 128 tokens the constants are an earlier fit's, which makes the better choices there (256 ids of the TinyLlama shape
// 2.03 ms, 2.06 by the newer one); the fast mode keeps that fit, and its tiles, so that its sums keep their order.
// Exact mode, by the earlier fit and so: 8B shape 10 ids 3.54 -> 3.35 ms, 40 4.21 -> 3.95, 90 5.76 -> 4.66; 1B 100 ids 1.27 -> 1.21.
//
// `max_splits`: ranges K may be cut into.  `row_step`: every matrix is a whole number of row_step rows.  `pair`: W1 and W3
// side by side in a tile (total_n counts both).
float planned_us(const Plan& p, int total_n, int K, int t_pad, bool lo, bool pair) {
    struct Cost {
        float launch, column, round, pair_round, rest;  // us, ns a column, us (the pair's: with SwiGLU), a last round's share at least
    };
    static constexpr Cost kCosts[3][2] = {{{4.9f, 7.4f, 4.7f, 4.9f, 0.67f}, {1.8f, 12.9f, 8.4f, 8.8f, 1.00f}},      // 128 x 128
                                          {{6.3f, 13.0f, 7.6f, 1.2f, 1.00f}, {16.4f, 21.3f, 9.6f, 7.5f, 0.94f}},    // 256 x 128
                                          {{0.0f, 20.5f, 5.8f, 18.4f, 1.00f}, {3.8f, 39.4f, 14.0f, 13.7f, 0.96f}}}; // blocks
    const Cost& c = kCosts[p.block() ? 2 : (p.fi == 4 ? 1 : 0)][lo ? 1 : 0];
    const int wgs = total_n / p.tile_rows() * p.token_tiles(t_pad, t_pad) * p.splits, left = wgs % compute_units();
    const float rounds = fmaxf(1.0f, wgs / compute_units() + (left > 0 ? c.rest + (1.0f - c.rest) * left / compute_units() : 0.0f));
    const float partials = p.splits > 1 ? 4.0f * p.splits * t_pad * total_n / 2.8e6f : 0.0f;
    return c.launch + rounds * (1e-3f * c.column * K / p.splits + (pair ? c.pair_round : c.round)) + partials;
}
Plan plan_gemm(int total_n, int K, int t_pad, int live, int max_splits, bool lo, int row_step, bool pair) {
    // `exact`, `fast`: padded tokens up to which a mode may be given the tile.  At 32 to 304 compute units, n to 300000 and K to
    // 32768 the model would give the exact mode no other; the fast mode's are those of the earlier fit.  launch_plan has the
    // kernels of this list.
    static constexpr struct {
        bool few;
        int fi, tj;
        int exact, fast;
    } kTiles[] = {{true, 1, 1, 256, 256}, {true, 1, 2, 0, 256}, {true, 1, 3, 128, 256}, {true, 2, 1, 256, 256},
                  {true, 2, 2, 256, 256}, {true, 2, 3, 256, 256}, {true, 2, 4, 0, 256},   {true, 4, 1, 256, 0},
                  {true, 4, 2, 256, 0},   {false, 2, 2, 256, 256}, {false, 4, 2, 256, 256}};
    Plan best = {false, 2, 2, 1};
    const bool wide_allowed = row_step % 256 == 0 && test_option(LPP_OPT_PREFILL_WIDE_TILES) != 0;
    if (t_pad > 256) {
        const int token_tiles = t_pad / 128;
        const bool wide = total_n / 256 * token_tiles >= compute_units() || (lo && total_n / 128 * token_tiles > compute_units());
        if (pair || (wide_allowed && wide)) best.fi = 4;
        while (2 * best.splits <= max_splits && total_n / best.tile_rows() * token_tiles * best.splits * 2 <= compute_units() &&
               K % (64 * 2 * best.splits) == 0 && K / (2 * best.splits) >= 512)
            best.splits *= 2;
        if (!wide_allowed) return best;
        // (the fast mode's results move by more than its bound when sums are cut elsewhere: there K stays cut as this rule cuts it)
        const int fast_splits = best.splits;
        float best_us = 1e30f;
        for (const auto& t : {Plan{false, 2, 2, 1}, Plan{false, 4, 2, 1}, Plan{false, 4, 4, 1}})
            for (int splits = 1; splits <= max_splits; splits *= 2) {
                if (splits > 1 && (K % (64 * splits) != 0 || K / splits < 512)) break;
                if (!lo && splits != fast_splits) continue;
                const Plan p = {t.few, t.fi, t.tj, splits};
                const float us = planned_us(p, total_n, K, t_pad, lo, pair);
                if (us < best_us) {
                    best_us = us;
                    best = p;
                }
            }
        return best;
    }
    struct Rates {
        float few, pipe, clocks;              // bytes and MFMA clocks a us
        float launch_few, launch_pipe, sums;  // us; of k_gemm_few's sums, a tile of 32 x 32
        float round;                          // what a round of workgroups costs whatever there is of it
        float weights, written, read;         // bytes a us: of weights, of partial products
    };
    // (kEarlier: by its clocks a tile's products take next to nothing, a thousandth of what they do, and no more than settle which
    // of two tiles of equal bytes it is.  The order of sums hangs on its choices, so they stay as they are.)
    static constexpr Rates kUpTo128 = {109e3f, 107e3f, 4.7e3f, 1.9f, 2.4f, 0.355f, 0.8f, 10.7e6f, 3.45e6f, 13.5e6f},
                           kEarlier = {57e3f, 88e3f, 5.7e6f, 1.9f, 1.9f, 0.0f, 0.87f, 3.9e6f, 2.5e6f, 5e6f};
    const bool earlier = !lo || t_pad > 128;
    const Rates& c = earlier ? kEarlier : kUpTo128;
    // A prompt and the same prompt filled up to 32, or beyond 128 tokens to 128, are summed alike: tokens count as whole columns
    // of those.
    const int counted = t_pad > 128 ? t_pad : (min(live, t_pad) + 31) / 32 * 32, columns = counted / 32;
    float best_us = 1e30f;
    for (const auto& t : kTiles) {
        const Plan p = {t.few, t.fi, t.tj, 1};
        const int rows = p.tile_rows(), tokens = p.tile_tokens(), token_tiles = p.token_tiles(t_pad, counted);
        if (row_step % rows != 0 || token_tiles * tokens > t_pad || (pair && t.fi == 1)) continue;
        if (t_pad > (lo ? t.exact : t.fast) || (earlier && counted % tokens != 0)) continue;
        if (!t.few && t.fi == 4 && !wide_allowed) continue;
        const int sent = min(tokens, 32 * ((columns + token_tiles - 1) / token_tiles));
        for (int splits = 1; splits <= max_splits; splits *= 2) {
            if (splits > 1 && (K % (64 * splits) != 0 || K / splits < 512)) continue;
            const int wgs = total_n / rows * token_tiles * splits, rounds = (wgs + compute_units() - 1) / compute_units();
            const float k = static_cast<float>(K) / splits, copies = lo ? 2.0f : 1.0f;
            const float bytes = k * 2.0f * (rows + copies * sent), clocks = k * copies * rows * sent / 1024.0f;
            const float turns = fmaxf(1.0f, c.round * rounds + (1.0f - c.round) * wgs / compute_units());
            const float sends = bytes / (t.few ? c.few : c.pipe), products = t.few ? 0.0f : clocks / c.clocks;
            const float busy = turns * (earlier ? sends + products : fmaxf(sends, products)), weights = 2.0f * total_n * K / c.weights;
            float us = (t.few ? c.launch_few + c.sums * t.fi * t.tj * rounds : c.launch_pipe + (earlier && t_pad <= 128 ? 1.0f : 0.0f)) +
                       fmaxf(busy, weights) + (earlier ? 0.0f : 0.01f * fminf(busy, weights));
            if (splits > 1) us += 4.0f * counted * total_n * (splits / c.written + (splits - 1) / c.read);
            if (us < best_us) {
                best_us = us;
                best = p;
                best.splits = splits;
            }
        }
    }
    return best;
}

// Floats that the partial products of one GEMM of a batch of t_pad tokens may take: at most eight ranges of 256 tokens, or one
// tile of 128 x 128 per compute unit, beyond 512 tokens one block of 256 x 256 (plan_gemm).  It goes by the batch alone: by the
// buffers that earlier calls have left, a batch would be cut, and so summed, differently behind a longer one.
size_t range_limit(const lpp_model* m, int t_pad) {
    const size_t few = t_pad < 256 ? t_pad : 256, cut = 8 * few * (m->cfg.dim + 2 * m->kv_dim);
    const size_t tiles = static_cast<size_t>(compute_units()) * (t_pad > pf::kSmallChunk ? 256 * 256 : 128 * 128);
    return t_pad > 256 && tiles > cut ? tiles : cut;
}

// The plan of a product of total_n rows; its partial products take `limit` floats at most.
Plan plan_product(int total_n, int K, int t_pad, int live, size_t limit, bool lo, int row_step) {
    const size_t stride = static_cast<size_t>(t_pad) * total_n;
    int most = 1;
    while (most < 8 && stride * 2 * most <= limit) most *= 2;
    return plan_gemm(total_n, K, t_pad, live, most, lo, row_step, false);
}
// The largest tile height that a matrix of n rows is a whole number of.
int tile_step(int n) { return n % 256 == 0 ? 256 : 128; }

// Floats of kBufPartials that chunks of up to t_pad tokens need: the partial products of the GEMM before (read by the
// kernel that follows it, so one area does for all of a layer's), or the gate and up projections where those are not fused.
// Up to 512 tokens that is range_limit.  Beyond, only the exact mode's plans go past it, at some shapes and lengths, so those
// lengths are asked (the fast mode keeps its cuts within a workgroup a compute unit).
size_t partial_floats(const lpp_model* m, int t_pad) {
    const int dim = m->cfg.dim, kv = m->kv_dim;
    const size_t pair = 2 * static_cast<size_t>(t_pad) * m->cfg.hidden_dim;
    const bool staged = test_option(LPP_OPT_PREFILL_STAGED_GEMM) != 0;
    size_t most = range_limit(m, t_pad < pf::kSmallChunk ? t_pad : pf::kSmallChunk);
    if (staged && m->pf_mode != LPP_PREFILL_FAST)
        for (int t = pf::kSmallChunk + pf::kTileTokens; t <= t_pad; t += pf::kTileTokens) {
            const size_t limit = range_limit(m, t);
            const int narrow = tile_step(dim) < tile_step(kv) ? tile_step(dim) : tile_step(kv);
            const struct { int n, k, step; } products[] = {{dim + 2 * kv, dim, narrow}, {2 * kv, dim, tile_step(kv)}, {dim, dim, tile_step(dim)},
                                                           {dim, m->cfg.hidden_dim, tile_step(dim)}};
            for (const auto& p : products) {
                const int splits = plan_product(p.n, p.k, t, t, limit, true, p.step).splits;
                const size_t floats = splits > 1 ? static_cast<size_t>(splits) * t * p.n : 0;
                if (floats > most) most = floats;
            }
        }
    const bool fused = staged && test_option(LPP_OPT_PREFILL_FUSED_FFN) != 0;
    return !fused && pair > most ? pair : most;
}

struct ScratchLayout {
    size_t offset[kBufAll];
    size_t total;
    size_t room;  // floats of kBufPartials
};
ScratchLayout scratch_layout(const lpp_model* m, int t_pad, size_t room) {
    const lpp_config& c = m->cfg;
    const size_t t = static_cast<size_t>(t_pad);
    ScratchLayout s = {};
    s.room = room;
    const size_t bytes[kBufAll] = {t * sizeof(int),
                                   t * c.dim * sizeof(float),
                                   t * c.dim * sizeof(float),
                                   t * m->kv_dim * sizeof(float),
                                   t * m->kv_dim * sizeof(float),
                                   s.room * sizeof(float),
                                   t * c.dim * sizeof(pf::half_t),
                                   t * c.dim * sizeof(pf::half_t),
                                   // the feed-forward activations, written while hi/lo are still being read
                                   t * c.hidden_dim * sizeof(pf::half_t),
                                   t * c.hidden_dim * sizeof(pf::half_t)};
    for (int i = 0; i < kBufAll; ++i) {
        s.offset[i] = s.total;
        s.total += (bytes[i] + 255) / 256 * 256;
    }
    return s;
}

// Tokens the buffers are made for where t_pad are needed: whole steps of 128 up to 512, of 512 beyond, so that prompts
// that grow from call to call seldom cost an allocation and the device-wide wait for the buffers given up.
int scratch_tokens(int t_pad) {
    const int step = t_pad <= pf::kSmallChunk ? pf::kTileTokens : pf::kSmallChunk;
    return (t_pad + step - 1) / step * step;
}

// What partial_floats goes by besides the tokens: buffers made under the same have room for every batch up to theirs.
int room_key(const lpp_model* m) {
    return 1 + (m->pf_mode != LPP_PREFILL_FAST) + 2 * (test_option(LPP_OPT_PREFILL_STAGED_GEMM) != 0) +
           4 * (test_option(LPP_OPT_PREFILL_FUSED_FFN) != 0) + 8 * (test_option(LPP_OPT_PREFILL_WIDE_TILES) != 0);
}

bool scratch_held(const lpp_model* m, int t_pad) {
    return m->pf_cap >= t_pad && (m->pf_room_key == room_key(m) || m->pf_room >= partial_floats(m, t_pad));
}

// Whether device memory has room for the buffers of t_pad tokens in the place of those the model holds: asked before those
// are given up, so that a model that lives with the smaller batch keeps its buffers from call to call.
bool scratch_fits(const lpp_model* m, int t_pad) {
    const int forced = test_option(LPP_OPT_PREFILL_ROOM);
    if (forced > 0 && t_pad > forced) return false;
    if (scratch_held(m, t_pad)) return true;
    size_t free_bytes = 0, all_bytes = 0;
    if (hipMemGetInfo(&free_bytes, &all_bytes) != hipSuccess) {
        (void)hipGetLastError();
        return true;  // (the allocation will say)
    }
    const size_t held = m->pf_cap > 0 ? scratch_layout(m, m->pf_cap, m->pf_room).total : 0;
    const int tokens = scratch_tokens(t_pad);
    return scratch_layout(m, tokens, partial_floats(m, tokens)).total <= free_bytes + held;
}

// `quiet`: an allocation that fails leaves lpp_last_error as it is (the caller has another way to go).  Buffers that are too
// small are made for as many tokens as they were, or more, so that a model that changes its mode from call to call settles.
lpp_status ensure_scratch(lpp_model* m, int t_pad, bool quiet = false) {
    if (scratch_held(m, t_pad)) return LPP_OK;
    const int needed = scratch_tokens(t_pad), before = m->pf_cap;
    prefill_release(m);
    const int forced = test_option(LPP_OPT_PREFILL_ROOM);
    ScratchLayout s = {};
    hipError_t e = hipErrorOutOfMemory;
    int tokens = before > needed ? before : needed;
    for (;; tokens = needed) {
        s = scratch_layout(m, tokens, partial_floats(m, tokens));
        if (forced >= 0 || t_pad <= -forced) e = hipMalloc(&m->pf_buf[kBufAll], s.total);
        if (e == hipSuccess || tokens == needed) break;
        (void)hipGetLastError();
    }
    if (e != hipSuccess) {
        (void)hipGetLastError();
        m->pf_buf[kBufAll] = nullptr;
        return quiet ? LPP_ERR_OOM : fail(LPP_ERR_OOM, "prefill buffers: hipMalloc(%zu) failed: %s", s.total, hipGetErrorString(e));
    }
    for (int i = 0; i < kBufAll; ++i) m->pf_buf[i] = static_cast<char*>(m->pf_buf[kBufAll]) + s.offset[i];
    m->pf_cap = tokens;
    m->pf_room = s.room;
    m->pf_room_key = room_key(m);
    return LPP_OK;
}

// Token tiles of k_gemm_pipe that a die's workgroups take at a time (PipeJob::band): four or the next larger divisor, bands of
// different lengths being slower than none (1280 ids in 4 + 4 + 2 tiles, 8B shape, fast mode: 24.5 -> 25.0 ms).  2048 ids,
// fast mode: 1B shape 5.81 -> 5.47 ms, 8B 37.6 -> 36.0, TinyLlama 6.70 -> 6.27; exact mode, paced by its MFMAs and LDS:
// 8B 53.8 -> 53.2, TinyLlama 9.53 -> 9.39, and up to 1408 ids between 2.5 % faster and 0.9 % slower, so not there.
// (By the counters, 1B shape, 2048 ids, fast: Wq+Wk+Wv has a fifth fewer L2 misses, 1.34 M -> 1.05 M, and goes from 46.0 to 39.6
// us; W1+W3, of four rounds of workgroups, has a fifth more, 2.88 M -> 3.44 M, and still goes from 184 to 169.)
int band_of(int token_tiles, bool lo) {
    if (token_tiles <= 4 || (lo && token_tiles < 12)) return token_tiles;
    int band = 4;
    while (token_tiles % band != 0) ++band;
    return band;
}

template <int kMode>
lpp_status launch_plan(const Plan& p, const pf::PipeJob& job_in, hipStream_t s) {
    pf::PipeJob job = job_in;
    job.band = band_of(job.token_tiles, job.xl != nullptr);
    if (p.block()) return job.xl != nullptr ? launch_block<kMode, true>(job, s) : launch_block<kMode, false>(job, s);
    if (!p.few) {
        if (p.fi == 4) return launch_pipe<4, 2, kMode>(job, s);
        return launch_pipe<2, 2, kMode>(job, s);
    }
    const bool lo = job.xl != nullptr;
    const int tile = 10 * p.fi + p.tj;
    if (lo && tile == 41) return launch_few<4, 1, kMode, true>(job, s);
    if (lo && tile == 42) return launch_few<4, 2, kMode, true>(job, s);
    if (!lo && tile == 24) return launch_few<2, 4, kMode, false>(job, s);
    if (tile == 21) return lo ? launch_few<2, 1, kMode, true>(job, s) : launch_few<2, 1, kMode, false>(job, s);
    if (tile == 22) return lo ? launch_few<2, 2, kMode, true>(job, s) : launch_few<2, 2, kMode, false>(job, s);
    if (tile == 23) return lo ? launch_few<2, 3, kMode, true>(job, s) : launch_few<2, 3, kMode, false>(job, s);
    if constexpr (kMode != 2) {  // (a pair has as many rows of either matrix in a tile)
        if (tile == 11) return lo ? launch_few<1, 1, kMode, true>(job, s) : launch_few<1, 1, kMode, false>(job, s);
        if (!lo && tile == 12) return launch_few<1, 2, kMode, false>(job, s);
        if (tile == 13) return lo ? launch_few<1, 3, kMode, true>(job, s) : launch_few<1, 3, kMode, false>(job, s);
    }
    return fail(LPP_ERR_STATE, "prefill GEMM: no kernel for a tile of %d x %d", p.tile_rows(), p.tile_tokens());
}

// Where the partial products of a split K go: `room` floats, of which a product may use `limit`.
struct Partials {
    float* at = nullptr;
    size_t limit = 0, room = 0;
};

// `area` (optional): room for partial products.  A product
// with too few output tiles for the compute units is cut along K into ranges, each multiplied by
// its own workgroups into the area: range z of matrix i lies at area.at + z * t_pad * (n_0 + n_1 +
// ..) + t_pad * (n_0 + .. + n_(i-1)), rows of n_i floats.  With `left_split` the caller adds the
// ranges itself (in order, in the kernel that reads the product next) and gets their number there;
// without it they are added to y here, in order.
lpp_status gemm(const Product* prods, int count, const pf::half_t* xh, const pf::half_t* xl, int K, int t_pad, bool accumulate,
                hipStream_t s, const Partials& area = {}, int* left_split = nullptr, bool remainder = true, int live = 0x7fffffff) {
    LPP_REQUIRE(count >= 1 && count <= 3 && t_pad > 0 && t_pad % 32 == 0 && K % 32 == 0, "prefill GEMM: %d products, K %d, T %d",
                count, K, t_pad);
    if (left_split != nullptr) *left_split = 1;
    int total_n = 0;
    int step = 256;  // largest tile height every matrix is a whole number of
    for (int i = 0; i < count; ++i) {
        LPP_REQUIRE(prods[i].n > 0 && prods[i].n % pf::kTileFeatures == 0, "prefill GEMM: n %d", prods[i].n);
        total_n += prods[i].n;
        if (tile_step(prods[i].n) < step) step = tile_step(prods[i].n);
    }
    const bool staged = K % pf::kPipeTripK == 0 && test_option(LPP_OPT_PREFILL_STAGED_GEMM) != 0;
    LPP_REQUIRE(staged || t_pad % pf::kTileTokens == 0, "prefill GEMM: T %d, K %d", t_pad, K);
    if (staged) {
        const size_t stride = static_cast<size_t>(t_pad) * total_n;
        live = live < t_pad ? live : t_pad;
        float* partials = area.at;
        const bool may_cut = partials != nullptr && (count == 1 || left_split != nullptr);
        const Plan plan = plan_product(total_n, K, t_pad, live, may_cut ? area.limit : 0, remainder, step);
        if (plan.splits > 1 && stride * plan.splits > area.room)
            return fail(LPP_ERR_STATE, "prefill GEMM: %zu floats of partial products, room for %zu", stride * plan.splits, area.room);
        const int tile = plan.tile_rows(), feature_tiles = total_n / tile, token_tiles = plan.token_tiles(t_pad, live), splits = plan.splits;
        pf::PipeJob job = {};
        int at = 0;
        size_t before = 0;
        for (int i = 0; i < 3; ++i) {
            const Product& p = prods[i < count ? i : count - 1];
            job.w[i] = static_cast<const pf::half_t*>(p.w);
            job.y[i] = splits > 1 ? partials + before : p.y;
            job.ldy[i] = p.n;
            job.first_tile[i] = i < count ? at : 0x7fffffff;
            if (i < count) {
                at += p.n / tile;
                before += static_cast<size_t>(t_pad) * p.n;
            }
        }
        job.xh = xh;
        job.xl = remainder ? xl : nullptr;  // (without: the kernels that neither fetch nor multiply the remainder)
        job.K = K;
        job.k_len = K / splits;
        job.split_stride = stride;
        job.feature_tiles = feature_tiles;
        job.token_tiles = token_tiles;
        job.live = live;
        job.rows = t_pad;
        job.groups = feature_tiles * splits;
        const bool add_in_kernel = accumulate && splits == 1;
        if (add_in_kernel) LPP_TRY(launch_plan<1>(plan, job, s));
        else LPP_TRY(launch_plan<0>(plan, job, s));
        if (splits > 1 && left_split != nullptr) {
            *left_split = splits;
        } else if (splits > 1) {
            if (accumulate)
                hipLaunchKernelGGL(pf::k_add_partials<true>, dim3(static_cast<unsigned>((stride / 4 + 255) / 256)), dim3(256), 0, s,
                                   prods[0].y, partials, splits, stride, stride);
            else
                hipLaunchKernelGGL(pf::k_add_partials<false>, dim3(static_cast<unsigned>((stride / 4 + 255) / 256)), dim3(256), 0, s,
                                   prods[0].y, partials, splits, stride, stride);
            LPP_CHECK_LAUNCH("k_add_partials");
        }
        return LPP_OK;
    }
    const bool large_tiles = (total_n / pf::kTileFeatures) * (t_pad / pf::kTileTokens) >= compute_units();
    const int tile = large_tiles ? pf::kTileFeatures : 64;
    // fragments straight from memory: one launch per matrix
    for (int i = 0; i < count; ++i) {
        const pf::half_t* wh = static_cast<const pf::half_t*>(prods[i].w);
        const dim3 grid(prods[i].n / tile, t_pad / tile);
        float* y = prods[i].y;
        const int ldy = prods[i].n;
        if (large_tiles) {
            if (accumulate) hipLaunchKernelGGL((pf::k_gemm<true, 2>), grid, dim3(256), 0, s, wh, xh, xl, y, K, ldy);
            else hipLaunchKernelGGL((pf::k_gemm<false, 2>), grid, dim3(256), 0, s, wh, xh, xl, y, K, ldy);
        } else {
            if (accumulate) hipLaunchKernelGGL((pf::k_gemm<true, 1>), grid, dim3(256), 0, s, wh, xh, xl, y, K, ldy);
            else hipLaunchKernelGGL((pf::k_gemm<false, 1>), grid, dim3(256), 0, s, wh, xh, xl, y, K, ldy);
        }
        LPP_CHECK_LAUNCH("k_gemm");
    }
    return LPP_OK;
}

// (remainders false: nobody reads lo after this norm, and the wide kernel leaves it unwritten)
lpp_status norm_split(float* x, const float* gain, pf::half_t* hi, pf::half_t* lo, int dim, int n, int t_pad, const float* partials,
                      int splits, size_t split_stride, hipStream_t s, bool remainders = true) {
    pf::half_t* lo_wide = remainders ? lo : nullptr;
#define LPP_NORM_WIDE(PER, SPLITS) \
    hipLaunchKernelGGL((pf::k_norm_split_wide<PER, SPLITS>), dim3(t_pad), dim3(256), 0, s, x, gain, hi, lo_wide, n, partials, split_stride)
#define LPP_NORM_WIDE_DIM(PER)          \
    switch (splits) {                   \
        case 0: LPP_NORM_WIDE(PER, 0); break; \
        case 2: LPP_NORM_WIDE(PER, 2); break; \
        case 4: LPP_NORM_WIDE(PER, 4); break; \
        default: LPP_NORM_WIDE(PER, 8); break; \
    }
    // (gemm() cuts K into 1, 2, 4 or 8 ranges)
    const bool wide = (dim == 1024 || dim == 2048 || dim == 4096) && (splits == 0 || splits == 2 || splits == 4 || splits == 8);
    if (wide && dim == 1024) {
        LPP_NORM_WIDE_DIM(1)
    } else if (wide && dim == 2048) {
        LPP_NORM_WIDE_DIM(2)
    } else if (wide) {
        LPP_NORM_WIDE_DIM(4)
    } else {
        hipLaunchKernelGGL(pf::k_norm_split, dim3(t_pad), dim3(256), 0, s, x, gain, hi, lo, dim, n, partials, splits, split_stride);
    }
#undef LPP_NORM_WIDE_DIM
#undef LPP_NORM_WIDE
    LPP_CHECK_LAUNCH("k_norm_split");
    return LPP_OK;
}

// (gemm() cuts K into 1, 2, 4 or 8 ranges)
lpp_status rope_scatter(const lpp_model* m, float* q, const float* qs, const float* ks, const float* vs, int layer, int pos0, int n,
                        int q_dim, int splits, size_t split_stride, hipStream_t s) {
    const auto kernel = splits == 1   ? &pf::k_rope_scatter<1>
                        : splits == 2 ? &pf::k_rope_scatter<2>
                        : splits == 4 ? &pf::k_rope_scatter<4>
                                      : &pf::k_rope_scatter<8>;
    hipLaunchKernelGGL(kernel, dim3((q_dim + 2 * m->kv_dim + 1023) / 1024, n), dim3(256), 0, s, q, qs, ks, vs, m->rope, m->key_cache,
                       m->value_cache, layer, pos0, q_dim, m->kv_dim, m->head_size, m->cfg.seq_len, split_stride);
    LPP_CHECK_LAUNCH("k_rope_scatter");
    return LPP_OK;
}

// (hi, lo)[t][u] = SwiGLU(W1 x[t], W3 x[t])[u] in one launch: the gate and the up projection of a
// feature share a workgroup, and the activation is applied to the accumulators.
lpp_status gate_up_swiglu(const void* w1, const void* w3, int hidden, const pf::half_t* xh, const pf::half_t* xl, int K, int t_pad,
                          pf::half_t* out_hi, pf::half_t* out_lo, hipStream_t s, bool remainder, int live) {
    pf::PipeJob job = {};
    job.w[0] = static_cast<const pf::half_t*>(w1);
    job.w[1] = static_cast<const pf::half_t*>(w3);
    job.w[2] = job.w[1];
    job.first_tile[0] = 0;
    job.first_tile[1] = job.first_tile[2] = 0x7fffffff;
    job.xh = xh;
    job.xl = remainder ? xl : nullptr;
    job.K = K;
    job.k_len = K;
    const Plan plan = plan_gemm(2 * hidden, K, t_pad, live, 1, remainder, hidden % 128 == 0 ? 256 : 128, true);
    job.feature_tiles = 2 * hidden / plan.tile_rows();  // half of a tile's rows from either matrix
    job.token_tiles = plan.token_tiles(t_pad, live);
    job.live = live;
    job.rows = t_pad;
    job.groups = job.feature_tiles;
    job.out_hi = out_hi;
    job.out_lo = out_lo;
    job.out_ld = hidden;
    return launch_plan<2>(plan, job, s);
}

template <int kHs, bool kLo, int kR, int kP>
lpp_status launch_attention_as(const lpp_model* m, const float* q, pf::half_t* hi, pf::half_t* lo, int layer, int pos0, int n, hipStream_t s) {
    constexpr int kLds = pf::AttentionShape<kHs, kR, kP>::kLdsBytes;
    static bool sized[64] = {};
    LPP_TRY(size_lds(reinterpret_cast<const void*>(&pf::k_attention_mfma<kHs, kLo, kR, kP>), kLds, sized));
    const int tokens = 32 * kR / m->gqa;
    hipLaunchKernelGGL((pf::k_attention_mfma<kHs, kLo, kR, kP>), dim3(m->cfg.n_kv_heads, (n + tokens - 1) / tokens), dim3(64 * kR * kP), kLds, s, q,
                       m->key_cache, m->value_cache, hi, lo, layer, pos0, m->cfg.dim, m->kv_dim, m->gqa, m->cfg.seq_len, n,
                       compute_units() / m->cfg.n_kv_heads);
    LPP_CHECK_LAUNCH("k_attention_mfma");
    return LPP_OK;
}
// Up to a tile of 32 rows per compute unit the longest walk is what counts, and eight wavefronts share it (heads of 128:
// four).  Up to two tiles, heads of 64: 2 x 2 would leave up to half of the compute units without a workgroup and walk the
// context in halves, 1 x 8 would be a second round of workgroups for most of them; 1 x 4 it is.  1B shape, exact mode,
// 257 ids behind 0 / 3000 / 7000, 1 x 8: 2.15 / 2.55 / 3.06 ms, 2 x 2: 2.10 / 2.67 / 3.42, 1 x 4: 2.09 / 2.46 / 2.91; 512 ids
// behind 7000: 3.71, 4.02, 3.62.  Above, the rows two wavefronts share count for more: 1024 ids, fast mode, behind 0: 2 x 2
// 3.13, 1 x 4 3.16; 640 ids behind 7000, exact, is the other way round (5.43, 5.12).  Heads of 128: 2 x 2 is the
// faster one throughout (six layers of the 8B shape's width, 257 ids behind 14000: 2.30 against 2.39; 1024: 4.30 against 4.86).
template <int kHs, bool kLo>
lpp_status launch_attention(const lpp_model* m, const float* q, pf::half_t* hi, pf::half_t* lo, int layer, int pos0, int n, hipStream_t s) {
    const int tokens = 32 / m->gqa, tiles = (n + tokens - 1) / tokens * m->cfg.n_kv_heads;
    if (tiles <= compute_units()) return launch_attention_as<kHs, kLo, 1, kHs == 64 ? 8 : 4>(m, q, hi, lo, layer, pos0, n, s);
    if constexpr (kHs == 64)
        if (tiles <= 2 * compute_units()) return launch_attention_as<kHs, kLo, 1, 4>(m, q, hi, lo, layer, pos0, n, s);
    return launch_attention_as<kHs, kLo, 2, 2>(m, q, hi, lo, layer, pos0, n, s);
}
lpp_status attention(const lpp_model* m, const float* q, pf::half_t* hi, pf::half_t* lo, int layer, int pos0, int n, bool remainders,
                     hipStream_t s) {
    if (m->head_size == 64)
        return remainders ? launch_attention<64, true>(m, q, hi, lo, layer, pos0, n, s) : launch_attention<64, false>(m, q, hi, lo, layer, pos0, n, s);
    return remainders ? launch_attention<128, true>(m, q, hi, lo, layer, pos0, n, s) : launch_attention<128, false>(m, q, hi, lo, layer, pos0, n, s);
}

// One chunk: tokens[0..n) at positions pos0 .. pos0 + n - 1; n <= kChunk.
lpp_status prefill_chunk(lpp_model* m, const int* tokens, int n, int pos0) {
    const lpp_config& c = m->cfg;
    const int dim = c.dim, kv = m->kv_dim, hidden = c.hidden_dim, hs = m->head_size;
    const int t_pad = padded_tokens(n);
    LPP_TRY(ensure_scratch(m, t_pad));
    hipStream_t s = stream();
    int* d_tokens = static_cast<int*>(m->pf_buf[kBufTokens]);
    float* x = static_cast<float*>(m->pf_buf[kBufX]);
    float* q = static_cast<float*>(m->pf_buf[kBufQ]);
    float* k = static_cast<float*>(m->pf_buf[kBufK]);
    float* v = static_cast<float*>(m->pf_buf[kBufV]);
    float* partials = static_cast<float*>(m->pf_buf[kBufPartials]);
    const Partials area = {partials, range_limit(m, t_pad), m->pf_room};
    pf::half_t* hi = static_cast<pf::half_t*>(m->pf_buf[kBufHi]);
    pf::half_t* lo = static_cast<pf::half_t*>(m->pf_buf[kBufLo]);
    LPP_HIP(hipMemcpyAsync(d_tokens, tokens, static_cast<size_t>(n) * sizeof(int), hipMemcpyHostToDevice, s));
    hipLaunchKernelGGL(pf::k_embed, dim3(n), dim3(256), 0, s, static_cast<const float*>(m->w[LPP_T_TOKEN_EMBEDDING]), d_tokens,
                       x, dim);
    LPP_CHECK_LAUNCH("k_embed");
    const size_t wb = sizeof(pf::half_t);
    auto layer_of = [&](int t, int l, size_t rows, size_t cols) {
        return static_cast<const char*>(m->w[t]) + static_cast<size_t>(l) * rows * cols * wb;
    };
    pf::half_t* hi2 = static_cast<pf::half_t*>(m->pf_buf[kBufHi2]);
    pf::half_t* lo2 = static_cast<pf::half_t*>(m->pf_buf[kBufLo2]);
    // LPP_PREFILL_EXACT: every product takes the activations as binary16 head + remainder.  LPP_PREFILL_FAST: the head
    // alone, in the staged kernels (what a GEMM sees of its input is then what the reference's own GPU GEMV sees,
    // matmul.cu:85-98; accumulation stays fp32).
    const bool exact = m->pf_mode != LPP_PREFILL_FAST;
    const bool fused_ffn = dim % pf::kPipeTripK == 0 && hidden % 128 == 0 && test_option(LPP_OPT_PREFILL_STAGED_GEMM) != 0 &&
                           test_option(LPP_OPT_PREFILL_FUSED_FFN) != 0;
    // Nobody reads a remainder when every GEMM of the chain is a staged one in the fast mode: the kernels that produce
    // activations then leave the remainders unwritten.  (The direct GEMM, taken for other shapes, always reads them.)
    const bool lean = !exact && fused_ffn;
    int pending = 0;  // ranges of the product before (W2's, then Wo's) still to be added to x
    for (int l = 0; l < c.n_layers; ++l) {
        // attention block, model.cpp:216-218
        LPP_TRY(norm_split(x, static_cast<const float*>(m->w[LPP_T_RMS_ATT]) + static_cast<size_t>(l) * dim, hi, lo, dim, n, t_pad, partials,
                           pending > 1 ? pending : 0, static_cast<size_t>(t_pad) * dim, s, !lean));
        // What a prefill leaves behind is the cache: the last layer needs its K and V rows only, and
        // nothing reads what the rest of that layer would compute.
        const bool last_layer = l == c.n_layers - 1;
        const Product qkv[3] = {{layer_of(LPP_T_WQ, l, dim, dim), q, dim}, {layer_of(LPP_T_WK, l, kv, dim), k, kv},
                                {layer_of(LPP_T_WV, l, kv, dim), v, kv}};
        const int q_dim = last_layer ? 0 : dim;
        int qkv_split = 1;
        LPP_TRY(gemm(qkv + (last_layer ? 1 : 0), last_layer ? 2 : 3, hi, lo, dim, t_pad, false, s, area, &qkv_split, exact, n));
        const size_t qkv_stride = static_cast<size_t>(t_pad) * (q_dim + 2 * kv);
        const float* qs = qkv_split > 1 ? partials : q;
        const float* ks = qkv_split > 1 ? partials + static_cast<size_t>(t_pad) * q_dim : k;
        const float* vs = qkv_split > 1 ? partials + static_cast<size_t>(t_pad) * (q_dim + kv) : v;
        LPP_TRY(rope_scatter(m, q, qs, ks, vs, l, pos0, n, q_dim, qkv_split, qkv_stride, s));
        if (last_layer) break;
        // (rows n .. t_pad of hi/lo are still the zeros k_norm_split wrote: the attention writes rows < n only)
        const bool matrix_cores = 32 % m->gqa == 0 && test_option(LPP_OPT_PREFILL_MFMA_ATTENTION) != 0;
        if (matrix_cores) {
            // (the fast mode rounds q and the softmax weights to binary16 as it rounds every GEMM input)
            LPP_TRY(attention(m, q, hi, lo, l, pos0, n, !lean, s));
        } else if (hs == 64)
            hipLaunchKernelGGL(pf::k_attention<8>, dim3((n + 3) / 4, c.n_kv_heads), dim3(256), 0, s, q, m->key_cache,
                               m->value_cache, hi, lo, l, pos0, dim, kv, hs, m->gqa, c.seq_len, n);
        else
            hipLaunchKernelGGL(pf::k_attention<16>, dim3((n + 3) / 4, c.n_kv_heads), dim3(256), 0, s, q, m->key_cache,
                               m->value_cache, hi, lo, l, pos0, dim, kv, hs, m->gqa, c.seq_len, n);
        LPP_CHECK_LAUNCH("k_attention");
        const Product wo = {layer_of(LPP_T_WO, l, dim, dim), x, dim};
        LPP_TRY(gemm(&wo, 1, hi, lo, dim, t_pad, true, s, area, &pending, exact, n));
        // feed-forward block, model.cpp:221-226
        LPP_TRY(norm_split(x, static_cast<const float*>(m->w[LPP_T_RMS_FFN]) + static_cast<size_t>(l) * dim, hi, lo, dim, n, t_pad, partials,
                           pending > 1 ? pending : 0, static_cast<size_t>(t_pad) * dim, s, !lean));
        if (fused_ffn) {
            LPP_TRY(gate_up_swiglu(layer_of(LPP_T_W1, l, hidden, dim), layer_of(LPP_T_W3, l, hidden, dim), hidden, hi, lo, dim, t_pad,
                                   hi2, lo2, s, exact, n));
        } else {
            float *gate = partials, *up = partials + static_cast<size_t>(t_pad) * hidden;
            const Product gate_up[2] = {{layer_of(LPP_T_W1, l, hidden, dim), gate, hidden}, {layer_of(LPP_T_W3, l, hidden, dim), up, hidden}};
            LPP_TRY(gemm(gate_up, 2, hi, lo, dim, t_pad, false, s, {}, nullptr, exact, n));
            hipLaunchKernelGGL(pf::k_swiglu_split, dim3((hidden + 255) / 256, t_pad), dim3(256), 0, s, gate, up, hi2, lo2, hidden, n);
            LPP_CHECK_LAUNCH("k_swiglu_split");
        }
        const Product w2 = {layer_of(LPP_T_W2, l, dim, hidden), x, dim};
        LPP_TRY(gemm(&w2, 1, hi2, lo2, hidden, t_pad, true, s, area, &pending, exact, n));
    }
    LPP_HIP(hipStreamSynchronize(s));
    return LPP_OK;
}

}  // namespace

void prefill_release(lpp_model* m) {
    lpp_free(m->pf_buf[kBufAll]);
    for (void*& p : m->pf_buf) p = nullptr;
    m->pf_cap = 0;
    m->pf_room = 0;
    m->pf_room_key = 0;
}

}  // namespace lpp

extern "C" {

lpp_status lpp_model_set_prefill_mode(lpp_model* m, int mode) {
    LPP_REQUIRE(m != nullptr && (mode == LPP_PREFILL_EXACT || mode == LPP_PREFILL_FAST), "lpp_model_set_prefill_mode: mode %d", mode);
    m->pf_mode = mode;
    return LPP_OK;
}

lpp_status lpp_prefill_supported(const lpp_model* m) {
    LPP_REQUIRE(m != nullptr, "lpp_prefill_supported: null model");
    const char* why = lpp::unsupported_reason(m);
    if (why != nullptr) return lpp::fail(LPP_ERR_UNSUPPORTED, "batched prefill unavailable: %s", why);
    return LPP_OK;
}

lpp_status lpp_prefill(lpp_model* m, const int* tokens, int n_tokens, int start_pos) {
    using namespace lpp;
    LPP_REQUIRE(m != nullptr && tokens != nullptr, "lpp_prefill: null argument");
    LPP_REQUIRE(n_tokens >= 0 && start_pos >= 0 && start_pos + n_tokens <= m->cfg.seq_len,
                "lpp_prefill: positions [%d, %d) outside [0, %d)", start_pos, start_pos + n_tokens, m->cfg.seq_len);
    for (int i = 0; i < n_tokens; ++i)
        LPP_REQUIRE(tokens[i] >= 0 && tokens[i] < m->cfg.vocab_size, "lpp_prefill: token %d at %d outside [0, %d)", tokens[i], i,
                    m->cfg.vocab_size);
    for (int t = 0; t < LPP_T_COUNT; ++t)
        if (!m->w_loaded[t]) return fail(LPP_ERR_STATE, "weight tensor %d has not been uploaded", t);
    LPP_TRY(lpp_prefill_supported(m));
    // Full chunks and a rest: 2048 tokens are the length that fills the device's rounds best.  (1B shape, exact: one chunk of
    // 2048 takes 7.2 ms, of 600 3.0, of 1270 5.2, so 2600 ids are better cut 2048 + 552 than into halves.)
    int each = n_tokens < pf::kChunk ? n_tokens : pf::kChunk;
    if (each > pf::kSmallChunk) {
        const int t_pad = padded_tokens(each);
        const lpp_status st = scratch_fits(m, t_pad) ? ensure_scratch(m, t_pad, true) : LPP_ERR_OOM;
        if (st == LPP_ERR_OOM) each = pf::kSmallChunk;
        else if (st != LPP_OK) return st;
    }
    for (int done = 0; done < n_tokens; done += each)
        LPP_TRY(prefill_chunk(m, tokens + done, n_tokens - done < each ? n_tokens - done : each, start_pos + done));
    return LPP_OK;
}

lpp_status lpp_prefill_gemm(float* d_y, const void* d_w, const float* d_x, int n, int k, int n_tokens, int accumulate) {
    using namespace lpp;
    LPP_REQUIRE(d_y && d_w && d_x, "lpp_prefill_gemm: null argument");
    LPP_REQUIRE(n_tokens > 0 && n_tokens % pf::kTileTokens == 0, "lpp_prefill_gemm: n_tokens %d not a positive multiple of %d",
                n_tokens, pf::kTileTokens);
    LPP_REQUIRE(n > 0 && n % pf::kTileFeatures == 0 && k > 0 && k % 32 == 0, "lpp_prefill_gemm: n %d k %d", n, k);
    hipStream_t s = stream();
    void* hi = nullptr;
    void* lo = nullptr;
    const size_t count = static_cast<size_t>(n_tokens) * k;
    LPP_TRY(lpp_malloc(&hi, count * sizeof(pf::half_t)));
    lpp_status st = lpp_malloc(&lo, count * sizeof(pf::half_t));
    if (st == LPP_OK) {
        hipLaunchKernelGGL(pf::k_split, dim3(static_cast<unsigned>((count + 255) / 256)), dim3(256), 0, s, d_x,
                           static_cast<pf::half_t*>(hi), static_cast<pf::half_t*>(lo), count);
        const Product one = {d_w, d_y, n};
        st = gemm(&one, 1, static_cast<pf::half_t*>(hi), static_cast<pf::half_t*>(lo), k, n_tokens, accumulate != 0, s);
        if (hipStreamSynchronize(s) != hipSuccess && st == LPP_OK) st = fail(LPP_ERR_HIP, "lpp_prefill_gemm: kernel failed");
    }
    lpp_free(hi);
    lpp_free(lo);
    return st;
}

}  // extern "C"

// ---------------------------------------------------------------------------
// The same product for callers that cannot allocate
// ---------------------------------------------------------------------------

namespace lpp {
namespace {

// Room for the binary16 head and remainder of the activations: kNoAllocElements each.
constexpr size_t kNoAllocElements = size_t{1} << 21;
static __device__ __align__(256) unsigned char scratch[2 * kNoAllocElements * sizeof(pf::half_t)];

// Device address of `scratch` per device.  In host code the array's name is only a handle
// for hipGetSymbolAddress; every device that loads the library holds its own copy.
constexpr int kMaxDevices = 64;
void* g_scratch_ptr[kMaxDevices] = {};

lpp_status scratch_address(void** out) {
    int device = -1;
    LPP_HIP(hipGetDevice(&device));
    if (device < 0 || device >= kMaxDevices) return fail(LPP_ERR_UNSUPPORTED, "device ordinal %d beyond %d", device, kMaxDevices - 1);
    if (g_scratch_ptr[device] == nullptr) {
        void* p = nullptr;
        LPP_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
        if (p == nullptr) return fail(LPP_ERR_HIP, "hipGetSymbolAddress returned no address for the prefill scratch");
        g_scratch_ptr[device] = p;
    }
    *out = g_scratch_ptr[device];
    return LPP_OK;
}

}  // namespace

namespace {
// What the set-up returned on each device: 0 not run yet, 1 done, 2 failed (message kept).
int g_setup_state[kMaxDevices] = {};
char g_setup_message[kMaxDevices][256] = {};

// (every tile of k_gemm_few that plan_gemm may give the exact mode for 128 or 256 tokens)
template <int kMode>
lpp_status size_few_for() {
    LPP_TRY((size_few<1, 1, kMode, true>()));
    LPP_TRY((size_few<2, 1, kMode, true>()));
    LPP_TRY((size_few<2, 2, kMode, true>()));
    LPP_TRY((size_few<4, 1, kMode, true>()));
    return size_few<4, 2, kMode, true>();
}

lpp_status run_scratch_setup() {
    LPP_TRY((size_pipe<4, 2, 0>()));
    LPP_TRY((size_pipe<4, 2, 1>()));
    LPP_TRY((size_pipe<2, 2, 0>()));
    LPP_TRY((size_pipe<2, 2, 1>()));
    LPP_TRY((size_block<0, true>()));
    LPP_TRY((size_block<1, true>()));
    LPP_TRY((size_few_for<0>()));
    LPP_TRY((size_few_for<1>()));
    void* p = nullptr;
    return scratch_address(&p);
}
}  // namespace

lpp_status prefill_gemm_scratch_setup() {
    // (everything the allocation-free entry point would otherwise set up on its first call: a caller under
    // graph capture finds it done)
    int device = -1;
    LPP_HIP(hipGetDevice(&device));
    if (device < 0 || device >= kMaxDevices) return fail(LPP_ERR_UNSUPPORTED, "device ordinal %d beyond %d", device, kMaxDevices - 1);
    const lpp_status st = run_scratch_setup();
    g_setup_state[device] = st == LPP_OK ? 1 : 2;
    if (st != LPP_OK) std::snprintf(g_setup_message[device], sizeof g_setup_message[device], "%s", lpp_last_error());
    return st;
}

// The set-up's outcome on the current device; runs it if this is the first call on the device.
static lpp_status prefill_gemm_scratch_status() {
    int device = -1;
    LPP_HIP(hipGetDevice(&device));
    if (device < 0 || device >= kMaxDevices) return fail(LPP_ERR_UNSUPPORTED, "device ordinal %d beyond %d", device, kMaxDevices - 1);
    if (g_setup_state[device] == 0) return prefill_gemm_scratch_setup();
    if (g_setup_state[device] == 2)
        return fail(LPP_ERR_HIP, "lpp_prefill_gemm_noalloc: set-up failed on this device: %s", g_setup_message[device]);
    return LPP_OK;
}

}  // namespace lpp

extern "C" {

lpp_status lpp_prefill_gemm_noalloc(float* d_y, const void* d_w, const float* d_x, int n, int k, int n_tokens, int accumulate) {
    using namespace lpp;
    LPP_REQUIRE(d_y && d_w && d_x, "lpp_prefill_gemm_noalloc: null argument");
    LPP_REQUIRE(n_tokens > 0 && n_tokens % pf::kTileTokens == 0, "lpp_prefill_gemm_noalloc: n_tokens %d not a positive multiple of %d",
                n_tokens, pf::kTileTokens);
    LPP_REQUIRE(n > 0 && n % pf::kTileFeatures == 0 && k > 0 && k % 32 == 0, "lpp_prefill_gemm_noalloc: n %d k %d", n, k);
    const size_t count = static_cast<size_t>(n_tokens) * k;
    LPP_REQUIRE(count <= kNoAllocElements, "lpp_prefill_gemm_noalloc: n_tokens * k = %zu exceeds the built-in scratch of %zu elements",
                count, kNoAllocElements);
    hipStream_t s = stream();
    LPP_TRY(prefill_gemm_scratch_status());
    void* base = nullptr;
    LPP_TRY(scratch_address(&base));
    pf::half_t* hi = static_cast<pf::half_t*>(base);
    pf::half_t* lo = hi + kNoAllocElements;
    hipLaunchKernelGGL(pf::k_split, dim3(static_cast<unsigned>((count + 255) / 256)), dim3(256), 0, s, d_x, hi, lo, count);
    LPP_CHECK_LAUNCH("k_split");
    const Product one = {d_w, d_y, n};
    return gemm(&one, 1, hi, lo, k, n_tokens, accumulate != 0, s);
}

}  // extern "C"
