// Causal attention of a prompt's rows in one launch, with the reference's
// rounding points (native/qwen3-tts-native/native/src/talker.cu:2772-2842,
// talker_kernels.cu:115-191,232-260: score to bf16, scaled score to bf16,
// probability to bf16, output to bf16; sums in fp32).
//
// A block of four waves takes 16 query rows of kHeads query heads that share a
// key/value head; the waves take the 32-key blocks up to the last row in turn
// (wave w: blocks w, w + 4, ...), so that the last rows' chain of blocks, the
// launch's critical path, is four times shorter than one wave's.
//   Sweep 1: scores by matrix cores, the running maximum and sum of
//     exponentials per lane (keys 8 apart), combined over lanes and waves.
//   Sweep 2: the scores again (cheaper than keeping a prompt's scores: keys
//     come from L2), each probability exp(s - max) * (1 / sum) rounded to
//     bf16, and the value products.
// Scores are formed transposed, S^T = K Q^T, with the key rows of two 16-row
// tiles dealt so that lane group g holds keys 8 g .. 8 g + 7 of its query:
// exactly the operand the value product takes, and exactly the 16-byte group
// in which the value cache holds 8 positions of one dimension.  So neither
// probabilities nor values move through LDS or a transposed copy.
//
// Bound by the exponentials (16 of them per lane, head and key block; q3_expf's
// bits: the hardware's exp2 with a first-order correction, 0.41 ulp rms against
// q3_expf's 0.30, saved 0.8 us of 16 at 512 rows) and the latency of a block's
// loads.  Per layer, 16 query and 8 key/value heads:
// 512 rows (score GEMM, softmax, value transpose, value GEMM) 60 us, 801 rows
// (per-row chains) 291 us before; now 16 and 32 us (33 rows, latency alone: 6 us).
#include "q3_common.hpp"
#include "q3_math.h"

namespace q3 {
namespace {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float floatx4_t __attribute__((ext_vector_type(4)));

constexpr int kDim = 128;
constexpr int kRows = 16;   // query rows of a block
constexpr int kKeys = 32;   // keys of a step
constexpr int kWaves = 4;

// Two floats to a pair of bf16 (nearest even) in one word, and back.
__device__ __forceinline__ unsigned pack(float lo, float hi) {
    typedef __bf16 pair_t __attribute__((ext_vector_type(2)));
    typedef float float_pair_t __attribute__((ext_vector_type(2)));
    return __builtin_bit_cast(unsigned, __builtin_convertvector(float_pair_t{lo, hi}, pair_t));
}
__device__ __forceinline__ float low_of(unsigned w) { return __uint_as_float(w << 16); }
__device__ __forceinline__ float high_of(unsigned w) { return __uint_as_float(w & 0xffff0000u); }

__device__ __forceinline__ bf16x8_t load8(const bf16_t* p) { return *reinterpret_cast<const bf16x8_t*>(p); }

template <int kHeads>
// Two waves a SIMD: unbounded, the compiler takes 1 us more (512 rows 16.9, now 16.2).
__global__ __launch_bounds__(64 * kWaves, 2) void prefill_attention_kernel(const bf16_t* qkv, int qkv_width,
                                                                         const bf16_t* key_cache,
                                                                         const bf16_t* value_cache, int value_stride,
                                                                         bf16_t* out, int rows, int query_heads,
                                                                         int key_value_heads, float scale) {
    __shared__ float max_lds[kWaves][kHeads][kRows], sum_lds[kWaves][kHeads][kRows];
    __shared__ __align__(16) float part[2][kHeads * 8 * 64 * 4];  // two waves' outputs, lane-major
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int m = lane & 15, group = lane >> 4;
    // the longest rows first: they are the launch's tail
    const int tile = (rows + kRows - 1) / kRows - 1 - static_cast<int>(blockIdx.x);
    const int q0 = tile * kRows;
    const int head0 = blockIdx.y * kHeads;
    const int kv_head = head0 / (query_heads / key_value_heads);
    const int kv_width = key_value_heads * kDim;
    const int query = q0 + m;  // this lane's query row (rows past the prompt repeat the last; not stored)
    const int last = min(q0 + kRows, rows) - 1;
    const int blocks = last / kKeys + 1;

    bf16x8_t qf[kHeads][4];
    {
        const bf16_t* q = qkv + static_cast<size_t>(min(query, rows - 1)) * qkv_width + head0 * kDim + 8 * group;
#pragma unroll
        for (int h = 0; h < kHeads; ++h)
#pragma unroll
            for (int kk = 0; kk < 4; ++kk) qf[h][kk] = load8(q + h * kDim + kk * 32);
    }
    // row i of key tile t holds key 8 (i >> 2) + 4 t + (i & 3) of the block
    const bf16_t* keys = key_cache + kv_head * kDim + 8 * group;
    const int key_row = 8 * (m >> 2) + (m & 3);
    auto load_keys = [&](int block, bf16x8_t (&kf)[2][4]) {
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            const bf16_t* k = keys + static_cast<size_t>(min(block * kKeys + key_row + 4 * t, rows - 1)) * kv_width;
#pragma unroll
            for (int kk = 0; kk < 4; ++kk) kf[t][kk] = load8(k + kk * 32);
        }
    };
    // s[h][2 t + w]: the scaled scores of keys block * 32 + 8 group + 4 t +
    // 2 w and the next, as bf16 (what they are rounded to)
    auto scores = [&](const bf16x8_t (&kf)[2][4], unsigned (&s)[kHeads][4]) {
#pragma unroll
        for (int h = 0; h < kHeads; ++h) {
            // two chains of two, not one of four: error of the 128 products'
            // sum, rms in 2^-24 of the sums', 0.84 against 1.00 (0.80 as the
            // exact kernels' tree; four products added: 0.80 too, but 8 us more
            // of 32 at 801 rows)
            floatx4_t acc[2];
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                floatx4_t half[2];
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                    half[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf[t][2 * i], qf[h][2 * i], floatx4_t{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
                    half[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf[t][2 * i + 1], qf[h][2 * i + 1], half[i], 0, 0, 0);
                }
                acc[t] = half[0] + half[1];
            }
#pragma unroll
            for (int t = 0; t < 2; ++t)
#pragma unroll
                for (int w = 0; w < 2; ++w) {
                    const unsigned dot = pack(acc[t][2 * w], acc[t][2 * w + 1]);
                    s[h][2 * t + w] = pack(low_of(dot) * scale, high_of(dot) * scale);
                }
        }
    };

    // ---- sweep 1 ----
    constexpr float kLowest = -3.402823466e+38f;
    float maximum[kHeads], sum[kHeads];
#pragma unroll
    for (int h = 0; h < kHeads; ++h) maximum[h] = kLowest, sum[h] = 0.f;
    bf16x8_t kf[2][4], vf[8];
    load_keys(wave, kf);
    for (int block = wave; block < blocks; block += kWaves) {
        unsigned s[kHeads][4];
        scores(kf, s);
        // the next block's keys (past the last: a repeat of the last row's,
        // unused) under this block's exponentials
        load_keys(block + kWaves, kf);
        const int visible = query - (block * kKeys + 8 * group);  // keys 0 .. visible of the lane's 8 count
#pragma unroll
        for (int h = 0; h < kHeads; ++h) {
            float top = maximum[h];
#pragma unroll
            for (int w = 0; w < 4; ++w) {
                top = 2 * w <= visible ? fmaxf(top, low_of(s[h][w])) : top;
                top = 2 * w + 1 <= visible ? fmaxf(top, high_of(s[h][w])) : top;
            }
            float add = sum[h] == 0.f ? 0.f : sum[h] * q3_expf_nonpositive(maximum[h] - top);
#pragma unroll
            for (int w = 0; w < 4; ++w) {
                add += 2 * w <= visible ? q3_expf_nonpositive(low_of(s[h][w]) - top) : 0.f;
                add += 2 * w + 1 <= visible ? q3_expf_nonpositive(high_of(s[h][w]) - top) : 0.f;
            }
            sum[h] = add;
            maximum[h] = top;
        }
    }
    // sweep 2's first keys and values, under the combination below
    const int groups8 = value_stride >> 3;
    const bf16_t* values = value_cache + static_cast<size_t>(kv_head) * groups8 * kDim * 8 + m * 8;
    // dims 16 d + m of positions 8 p .. 8 p + 7, p = 4 block + group
    auto load_values = [&](int block) {
        const bf16_t* v = values + static_cast<size_t>(min(block * 4 + group, groups8 - 1)) * kDim * 8;
#pragma unroll
        for (int d = 0; d < 8; ++d) vf[d] = load8(v + d * 16 * 8);
    };
    load_keys(wave, kf);
    load_values(wave);
    // over the four lanes of a query, then over the waves
#pragma unroll
    for (int h = 0; h < kHeads; ++h) {
#pragma unroll
        for (int d = 16; d < 64; d <<= 1) {
            const float other_max = __shfl_xor(maximum[h], d, 64), other_sum = __shfl_xor(sum[h], d, 64);
            const float top = fmaxf(maximum[h], other_max);
            const float mine = sum[h] == 0.f ? 0.f : sum[h] * q3_expf_nonpositive(maximum[h] - top);
            const float theirs = other_sum == 0.f ? 0.f : other_sum * q3_expf_nonpositive(other_max - top);
            sum[h] = mine + theirs;
            maximum[h] = top;
        }
        if (group == 0) max_lds[wave][h][m] = maximum[h], sum_lds[wave][h][m] = sum[h];
    }
    __syncthreads();
    float inverse[kHeads];
#pragma unroll
    for (int h = 0; h < kHeads; ++h) {
        float top = max_lds[0][h][m];
#pragma unroll
        for (int w = 1; w < kWaves; ++w) top = fmaxf(top, max_lds[w][h][m]);
        float total = 0.f;
#pragma unroll
        for (int w = 0; w < kWaves; ++w) {
            const float part_sum = sum_lds[w][h][m];
            total += part_sum == 0.f ? 0.f : part_sum * q3_expf_nonpositive(max_lds[w][h][m] - top);
        }
        maximum[h] = top;
        inverse[h] = 1.0f / total;
    }

    // ---- sweep 2 ----
    floatx4_t acc[kHeads][8];  // [dimension tile]: dims 16 tile + 4 group + r of query m
#pragma unroll
    for (int h = 0; h < kHeads; ++h)
#pragma unroll
        for (int d = 0; d < 8; ++d) acc[h][d] = floatx4_t{0.f, 0.f, 0.f, 0.f};
    for (int block = wave; block < blocks; block += kWaves) {
        unsigned s[kHeads][4];
        scores(kf, s);
        load_keys(block + kWaves, kf);
        const int visible = query - (block * kKeys + 8 * group);
        bf16x8_t pf[kHeads];
#pragma unroll
        for (int h = 0; h < kHeads; ++h) {
            unsigned pw[4];
#pragma unroll
            for (int w = 0; w < 4; ++w) {
                const float lo = q3_expf_nonpositive(low_of(s[h][w]) - maximum[h]) * inverse[h];
                const float hi = q3_expf_nonpositive(high_of(s[h][w]) - maximum[h]) * inverse[h];
                pw[w] = pack(2 * w <= visible ? lo : 0.f, 2 * w + 1 <= visible ? hi : 0.f);
            }
            pf[h] = __builtin_bit_cast(bf16x8_t, uint4{pw[0], pw[1], pw[2], pw[3]});
        }
        if (block * kKeys + kKeys > rows) {
            // positions past the prompt hold anything (another utterance's
            // values, NaN): zero them, as a zero probability would not
            const int valid = rows - (block * 4 + group) * 8;
#pragma unroll
            for (int d = 0; d < 8; ++d) {
                uint4 bits = __builtin_bit_cast(uint4, vf[d]);
                unsigned* word = &bits.x;
#pragma unroll
                for (int w = 0; w < 4; ++w)
                    word[w] = valid >= 2 * w + 2 ? word[w] : valid == 2 * w + 1 ? word[w] & 0xffffu : 0u;
                vf[d] = __builtin_bit_cast(bf16x8_t, bits);
            }
        }
#pragma unroll
        for (int h = 0; h < kHeads; ++h)
#pragma unroll
            for (int d = 0; d < 8; ++d) acc[h][d] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf[d], pf[h], acc[h][d], 0, 0, 0);
        load_values(block + kWaves);
    }
    // waves 2 and 3 into waves 0 and 1, wave 1 into wave 0
    auto put = [&](float* to) {
#pragma unroll
        for (int h = 0; h < kHeads; ++h)
#pragma unroll
            for (int d = 0; d < 8; ++d) *reinterpret_cast<floatx4_t*>(to + ((h * 8 + d) * 64 + lane) * 4) = acc[h][d];
    };
    auto take = [&](const float* from) {
#pragma unroll
        for (int h = 0; h < kHeads; ++h)
#pragma unroll
            for (int d = 0; d < 8; ++d) acc[h][d] += *reinterpret_cast<const floatx4_t*>(from + ((h * 8 + d) * 64 + lane) * 4);
    };
    if (wave >= 2) put(part[wave - 2]);
    __syncthreads();
    if (wave < 2) take(part[wave]);
    __syncthreads();
    if (wave == 1) put(part[0]);
    __syncthreads();
    if (wave != 0) return;
    take(part[0]);
    if (query >= rows) return;
    bf16_t* o = out + static_cast<size_t>(query) * query_heads * kDim + head0 * kDim + 4 * group;
#pragma unroll
    for (int h = 0; h < kHeads; ++h)
#pragma unroll
        for (int d = 0; d < 8; ++d) {
            const uint2 r{pack(acc[h][d][0], acc[h][d][1]), pack(acc[h][d][2], acc[h][d][3])};
            *reinterpret_cast<uint2*>(o + h * kDim + 16 * d) = r;
        }
}

}  // namespace

hipError_t launch_prefill_attention(const bf16_t* qkv, int qkv_width, const bf16_t* key_cache, const bf16_t* value_cache,
                                    int value_stride, bf16_t* out, int rows, int query_heads, int key_value_heads,
                                    int head_dimension, hipStream_t stream) {
    if (qkv == nullptr || key_cache == nullptr || value_cache == nullptr || out == nullptr || rows <= 0 ||
        key_value_heads <= 0 || query_heads <= 0 || query_heads % key_value_heads != 0 || head_dimension != kDim ||
        value_stride % 8 != 0 || value_stride < rows || qkv_width % 8 != 0 ||
        qkv_width < (query_heads + 2 * key_value_heads) * kDim) {
        return hipErrorInvalidValue;
    }
    const float scale = 1.0f / sqrtf(static_cast<float>(head_dimension));
    const int tiles = (rows + kRows - 1) / kRows;
    // two heads of a key/value head share its key and value loads, once blocks
    // of one head would outnumber the 256 CUs; below, latency alone counts and
    // a block of one head has half the exponentials in its chain (33 rows, two
    // heads 10.8 us a layer).  A head's arithmetic is the same either way.
    if (query_heads / key_value_heads % 2 == 0 && tiles * query_heads > 256) {
        prefill_attention_kernel<2><<<dim3(tiles, query_heads / 2), 64 * kWaves, 0, stream>>>(
            qkv, qkv_width, key_cache, value_cache, value_stride, out, rows, query_heads, key_value_heads, scale);
    } else {
        prefill_attention_kernel<1><<<dim3(tiles, query_heads), 64 * kWaves, 0, stream>>>(
            qkv, qkv_width, key_cache, value_cache, value_stride, out, rows, query_heads, key_value_heads, scale);
    }
    return hipGetLastError();
}

}  // namespace q3
