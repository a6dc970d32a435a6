// Kernels of the speech-tokenizer decoder (reference:
// native/qwen3-tts-native-codec/native/src/codec_state.cu, cited CS:line).
//
// The reference runs cuBLAS SGEMM plus one elementwise kernel per operation.
// Here the convolutions are fp32 matrix-core kernels (conv_gemm.hip) that read
// their input in place and whose epilogue applies bias, GELU, the residual and
// the following SnakeBeta, writing the next layer's input directly.  This file
// holds the transformer's 1..4-row products (RMSNorm fused) and the rest; blockIdx.z (or .y) is the stream where
// a batch shares a launch.
#include "codec.hpp"

#include "../q3_math.h"

#include <algorithm>

namespace q3c {

namespace {

__device__ __forceinline__ float wave_sum(float v) {
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}

// The wave's sums of kCount (a power of two) values: sum q in the lanes whose
// lane / (64 / kCount) is q, added in wave_sum's pairs, so with its bits.  A
// step halves the values a lane still carries: 7 exchanges for four sums, not
// 24, and 10 for eight.
template <int kCount>
__device__ __forceinline__ float wave_sums(float (&v)[kCount]) {
    const int lane = threadIdx.x & 63;
    int o = 32;
#pragma unroll
    for (int n = kCount / 2; n > 0; n >>= 1, o >>= 1) {
        const bool upper = lane & o;
#pragma unroll
        for (int i = 0; i < n; ++i) {
            const float keep = upper ? v[i + n] : v[i], give = upper ? v[i] : v[i + n];
            v[i] = keep + __shfl_xor(give, o, 64);
        }
    }
    float sum = v[0];
    for (; o > 0; o >>= 1) sum += __shfl_xor(sum, o, 64);
    return sum;
}

__device__ __forceinline__ float wave_max(float v) {
    for (int o = 32; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o, 64));
    return v;
}

__device__ __forceinline__ float4 load4(const float* p) { return *reinterpret_cast<const float4*>(p); }

inline unsigned blocks_for(size_t count, unsigned threads = 256) {
    const size_t b = (count + threads - 1) / threads;
    return (unsigned)std::min<size_t>(std::max<size_t>(b, 1), 65535u * 16);
}

// `p` of the first stream, for stream s
template <typename T>
__device__ __forceinline__ T* of_stream(T* p, const Streams& st, int s) {
    return s == 0 ? p : reinterpret_cast<T*>(reinterpret_cast<uintptr_t>(p) + st.delta[s]);
}

// ---------------------------------------------------------------------------
// Rows GEMV for 1..4 rows (transformer projections, RVQ projection, causal
// pre-convolution).  One wave computes one output channel of one stream
// (blockIdx.y): its lanes hold the rows in registers (float4 at k = 256 * c +
// 4 * lane, read from L2), apply RMSNorm there when asked (CS:414-434: each wave reduces the
// row's squares itself), stream each channel's weight row with float4 loads
// and finish with butterfly sums.  No LDS and no barrier: the launch's
// latency is one weight read plus one reduction (two with the norm), so the
// rows' sums travel together (wave_sums) and the epilogue's operands are
// requested beside the weights (a 1-frame packet 590 -> 545 us,
// 4 frames 757 -> 737 us, six streams 2235 -> 2189 us).  Four channels a
// block: one wave a block cost the packet about 5 us more.  Matrix-core tiles (16 rows, 4 used) were
// slower here: 512 x 1024 3.3 -> 5.6 us, gate/up 5.2 -> 6.9 us.
// kRows: 1, 2 or 4, the least that holds the packet's rows.
// ---------------------------------------------------------------------------
constexpr int kMaxRows = 4;

constexpr int kGemvWaves = 4;

template <int kChunks, int kRows, bool kPair>
__global__ __launch_bounds__(64 * kGemvWaves) void rows_gemv_kernel(RowsGemvArgs g) {
    constexpr int kSums = kPair ? 2 * kRows : kRows, kLanes = 64 / kSums;
    const int lane = threadIdx.x & 63;
    const int ch = blockIdx.x * kGemvWaves + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const float* rows_x = of_stream(g.x, g.streams, blockIdx.y);
    // the channel's weight row(s) first: the longest-latency reads
    float4 wa[kChunks], wb[kPair ? kChunks : 1];
#pragma unroll
    for (int c = 0; c < kChunks; ++c) wa[c] = load4(g.w + (size_t)ch * g.k + c * 256 + lane * 4);
    if constexpr (kPair) {
#pragma unroll
        for (int c = 0; c < kChunks; ++c) wb[c] = load4(g.w + (size_t)(g.n + ch) * g.k + c * 256 + lane * 4);
    }
    float4 x[kRows][kChunks];
#pragma unroll
    for (int r = 0; r < kRows; ++r) {
        const int rr = min(r, g.rows - 1);
#pragma unroll
        for (int c = 0; c < kChunks; ++c) x[r][c] = load4(rows_x + (size_t)rr * g.ldx + c * 256 + lane * 4);
    }
    // sum q (of row q) ends in the lanes from q * kLanes on, the first of
    // which finishes it; a pair's second half follows in the upper lanes
    const int row = lane / kLanes;
    const size_t at = (size_t)min(row, g.rows - 1) * g.ldo + ch;
    const bool residual_add = !kPair && g.epilogue == kRowsScaledResidual;
    const float bias = !kPair && g.bias ? g.bias[ch] : 0.f;
    const float scale = residual_add ? g.scale[ch] : 0.f;
    const float residual = residual_add ? of_stream(g.residual, g.streams, blockIdx.y)[at] : 0.f;
    if (g.norm) {
        float4 nw[kChunks];
#pragma unroll
        for (int c = 0; c < kChunks; ++c) nw[c] = load4(g.norm + c * 256 + lane * 4);
        float square[kRows];
#pragma unroll
        for (int r = 0; r < kRows; ++r) {
            float sq = 0.f;
#pragma unroll
            for (int c = 0; c < kChunks; ++c) {
                sq = fmaf(x[r][c].x, x[r][c].x, sq);
                sq = fmaf(x[r][c].y, x[r][c].y, sq);
                sq = fmaf(x[r][c].z, x[r][c].z, sq);
                sq = fmaf(x[r][c].w, x[r][c].w, sq);
            }
            square[r] = sq;
        }
        const float inverse = 1.0f / sqrtf(wave_sums(square) / (float)g.k + 1.0e-5f);
#pragma unroll
        for (int r = 0; r < kRows; ++r) {
            const float by = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(inverse), r * (64 / kRows)));
#pragma unroll
            for (int c = 0; c < kChunks; ++c) {
                x[r][c].x = x[r][c].x * by * nw[c].x;
                x[r][c].y = x[r][c].y * by * nw[c].y;
                x[r][c].z = x[r][c].z * by * nw[c].z;
                x[r][c].w = x[r][c].w * by * nw[c].w;
            }
        }
    }
    if (g.advance_position && ch == 0 && lane == 0)
        *of_stream(g.advance_position, g.streams, blockIdx.y) += g.advance_by;

    float sums[kSums];
    auto dot_row = [&](const float4* wv, int r) {
        float s = 0.f;
#pragma unroll
        for (int c = 0; c < kChunks; ++c) {
            s = fmaf(wv[c].x, x[r][c].x, s);
            s = fmaf(wv[c].y, x[r][c].y, s);
            s = fmaf(wv[c].z, x[r][c].z, s);
            s = fmaf(wv[c].w, x[r][c].w, s);
        }
        return s;
    };
#pragma unroll
    for (int r = 0; r < kRows; ++r) {
        sums[r] = dot_row(wa, r);
        if constexpr (kPair) sums[kRows + r] = dot_row(wb, r);
    }
    const float va = wave_sums(sums);
    float v;
    if constexpr (kPair) {
        const float vb = __shfl_xor(va, 32, 64);
        v = (va / (1.0f + q3_expf(-va))) * vb;  // CS:687-698
    } else {
        v = g.bias ? va + bias : va;
        if (residual_add) v = residual + v * scale;
    }
    if (lane % kLanes == 0 && row < g.rows) of_stream(g.out, g.streams, blockIdx.y)[at] = v;
}

// ---------------------------------------------------------------------------
// Transformer attention of one packet (CS:464-494 RoPE, CS:496-566 sliding
// attention).  One block per (head, frame, stream).  Each block rotates the
// packet's own keys itself (so no block reads a ring slot another block writes
// in the same launch), takes older keys and values from the ring, and follows
// the reference's per-head loop: scores, max, exponentials, denominator, the
// per-term probabilities and the value sum.  Frame 0's block appends the
// packet's keys and values to the ring.
//
// Latency-bound (16 heads x 1..4 frames): scores split each key's 64 products
// over two lanes, the denominator is a wave's tree and the values run as four
// partial sums over 18 positions each; cosines and sines come from the
// frontend instead of powf, sinf and cosf here.  9 us a launch before,
// 6.8 now (four frames).
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void codec_attention_kernel(const float* qkv, int frames,
                                                              const unsigned long long* position,
                                                              const float* rotations, float* kv_k, float* kv_v,
                                                              float* out, Streams streams) {
    __shared__ float q_s[64];
    __shared__ float k_s[kWindow][65];
    __shared__ float v_s[kWindow][64];
    __shared__ float p_s[kWindow];
    __shared__ float part_s[4][64];
    const int head = blockIdx.x, f = blockIdx.y, stream = blockIdx.z;
    const int tid = threadIdx.x;
    qkv = of_stream(qkv, streams, stream);
    rotations = of_stream(rotations, streams, stream);
    const unsigned long long pos = *of_stream(position, streams, stream);
    const unsigned long long me = pos + (unsigned long long)f;
    const unsigned long long first = me + 1 > (unsigned long long)kWindow ? me + 1 - kWindow : 0ull;
    const int count = (int)(me - first + 1);
    const int old_rows = (int)(pos - first);  // window rows before the packet
    float* ring_k = of_stream(kv_k, streams, stream) + (size_t)head * kKvSlots * 64;
    float* ring_v = of_stream(kv_v, streams, stream) + (size_t)head * kKvSlots * 64;
    const int first_slot = (int)(first % kKvSlots);
    // the packet's frames 0..f, rotate-half pairs (d, d + 32); frame 0's block
    // also appends every frame's row to the ring
    if (tid < 128 && (tid >> 5) < frames) {
        const int g = tid >> 5, d = tid & 31;
        const float* row = qkv + (size_t)g * 3 * 1024 + head * 64;
        const float cosine = rotations[(g * 32 + d) * 2], sine = rotations[(g * 32 + d) * 2 + 1];
        const float k1 = row[1024 + d], k2 = row[1024 + d + 32];
        const float v1 = row[2048 + d], v2 = row[2048 + d + 32];
        const float r1 = k1 * cosine - k2 * sine, r2 = k2 * cosine + k1 * sine;
        if (g <= f) {
            const int j = old_rows + g;
            k_s[j][d] = r1;
            k_s[j][d + 32] = r2;
            v_s[j][d] = v1;
            v_s[j][d + 32] = v2;
        }
        if (g == f) {
            const float q1 = row[d], q2 = row[d + 32];
            q_s[d] = q1 * cosine - q2 * sine;
            q_s[d + 32] = q2 * cosine + q1 * sine;
        }
        if (f == 0) {
            const int slot = (int)((pos + (unsigned long long)g) % kKvSlots);
            ring_k[slot * 64 + d] = r1;
            ring_k[slot * 64 + d + 32] = r2;
            ring_v[slot * 64 + d] = v1;
            ring_v[slot * 64 + d + 32] = v2;
        }
    }
    for (int idx = tid; idx < old_rows * 16; idx += 256) {  // float4 per thread
        const int j = idx >> 4, d = (idx & 15) * 4;
        int slot = first_slot + j;
        slot -= slot >= kKvSlots ? kKvSlots : 0;
        const float4 kk = load4(ring_k + slot * 64 + d), vv = load4(ring_v + slot * 64 + d);
        k_s[j][d] = kk.x, k_s[j][d + 1] = kk.y, k_s[j][d + 2] = kk.z, k_s[j][d + 3] = kk.w;
        *reinterpret_cast<float4*>(&v_s[j][d]) = vv;
    }
    __syncthreads();
    // key j = tid / 2: dims 32 (tid & 1) .. + 31, four chains
    float score = -3.402823466e+38f;
    {
        const int j = min(tid >> 1, count - 1), d0 = 32 * (tid & 1);
        float sc[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int d = 0; d < 32; d += 4)
#pragma unroll
            for (int i = 0; i < 4; ++i) sc[i] = fmaf(q_s[d0 + d + i], k_s[j][d0 + d + i], sc[i]);
        float dot = (sc[0] + sc[1]) + (sc[2] + sc[3]);
        dot += __shfl_xor(dot, 1, 64);
        if ((tid >> 1) < count) score = dot * 0.125f;
    }
    // keys lie in waves 0..2: max and denominator over them
    __shared__ float wmax[4], wsum[4];
    const float m = wave_max(score);
    if ((tid & 63) == 0) wmax[tid >> 6] = m;
    __syncthreads();
    const float maximum = fmaxf(fmaxf(wmax[0], wmax[1]), fmaxf(wmax[2], wmax[3]));
    const float e = (tid >> 1) < count ? q3_expf(score - maximum) : 0.f;
    const float total = wave_sum((tid & 1) == 0 ? e : 0.f);
    if ((tid & 63) == 0) wsum[tid >> 6] = total;
    __syncthreads();
    const float denominator = (wsum[0] + wsum[1]) + (wsum[2] + wsum[3]);
    if ((tid & 1) == 0 && (tid >> 1) < count) p_s[tid >> 1] = e / denominator;  // the reference's per-term probability
    __syncthreads();
    {
        const int d = tid & 63, quarter = tid >> 6;
        const int j0 = quarter * (kWindow / 4), j1 = min(count, j0 + kWindow / 4);
        float result = 0.f;
#pragma unroll 6
        for (int j = j0; j < j1; ++j) result = fmaf(p_s[j], v_s[j][d], result);
        part_s[quarter][d] = result;
    }
    __syncthreads();
    if (tid < 64)
        of_stream(out, streams, stream)[(size_t)f * 1024 + head * 64 + tid] =
            (part_s[0][tid] + part_s[1][tid]) + (part_s[2][tid] + part_s[3][tid]);
}

// ---------------------------------------------------------------------------
// Frontend codebook gather (CS:322-342) and history copies.
// ---------------------------------------------------------------------------
struct FrontendTables {
    const float* emb[kCodebooks];
    const float* usage[kCodebooks];
};

// Segment blockIdx.y of stream blockIdx.z, chunk `block` of `blocks`.
__device__ void copy_segment_chunk(const CopySegment* seg, const Streams& streams, int block, int blocks) {
    const CopySegment sg = seg[blockIdx.y];
    const unsigned n4 = sg.floats >> 2;
    const float4* src = reinterpret_cast<const float4*>(of_stream(sg.src, streams, blockIdx.z));
    float4* dst = reinterpret_cast<float4*>(of_stream(sg.dst, streams, blockIdx.z));
    for (unsigned i = block * 256 + threadIdx.x; i < n4; i += blocks * 256) dst[i] = src[i];
}

// blockIdx.y = segment, blockIdx.z = stream; on segment row 0 the first
// `frames` blocks also gather frame blockIdx.x's codebook entries (all 16
// lookups issued at once), and on row 1 they form the frame's RoPE angles.
__global__ __launch_bounds__(256) void codec_frontend_kernel(const uint16_t* codes, int frames, FrontendTables t,
                                                             float* x, const unsigned long long* position,
                                                             float* rotations, const CopySegment* seg,
                                                             Streams streams) {
    if (blockIdx.y == 1 && (int)blockIdx.x < frames && threadIdx.x < 32) {
        const int f = blockIdx.x, d = threadIdx.x;
        const unsigned long long at = *of_stream(position, streams, blockIdx.z) + (unsigned long long)f;
        const float angle = (float)at * (1.0f / powf(10000.0f, (float)(2 * d) / 64.0f));
        float* to = of_stream(rotations, streams, blockIdx.z) + (f * 32 + d) * 2;
        to[0] = cosf(angle);
        to[1] = sinf(angle);
    }
    if (blockIdx.y == 0 && (int)blockIdx.x < frames) {
        codes += blockIdx.z * (kMaxFrames * kCodebooks);
        x = of_stream(x, streams, blockIdx.z);
        const int f = blockIdx.x, d = threadIdx.x;
        int code[kCodebooks];
        float usage[kCodebooks], emb[kCodebooks];
#pragma unroll
        for (int cb = 0; cb < kCodebooks; ++cb) {
            // codes beyond the 2048-entry codebooks are clamped so a corrupt
            // device frame cannot read outside the table
            code[cb] = min((int)codes[f * kCodebooks + cb], 2047);
        }
#pragma unroll
        for (int cb = 0; cb < kCodebooks; ++cb) {
            usage[cb] = t.usage[cb][code[cb]];
            emb[cb] = t.emb[cb][(size_t)code[cb] * 256 + d];
        }
        float acoustic = 0.f;
#pragma unroll
        for (int cb = 0; cb < kCodebooks; ++cb) {
            const float value = emb[cb] / fmaxf(usage[cb], 1.0e-5f);
            if (cb == 0) {
                x[f * 512 + d] = value;
            } else {
                acoustic = cb == 1 ? value : acoustic + value;
            }
        }
        x[f * 512 + 256 + d] = acoustic;
    }
    copy_segment_chunk(seg, streams, blockIdx.x, gridDim.x);
}

__global__ __launch_bounds__(256) void copy_segments_kernel(const CopySegment* seg, Streams streams) {
    copy_segment_chunk(seg, streams, blockIdx.x, gridDim.x);
}

// ---------------------------------------------------------------------------
// ConvNeXt depthwise causal convolution (CS:730-756) + LayerNorm (CS:778-808):
// one block per position, 4 channels per thread.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void dwconv_layernorm_kernel(const float* ext, const float* w, const float* b,
                                                               const float* ln_w, const float* ln_b, float* out,
                                                               Streams streams) {
    __shared__ float red[4];
    ext = of_stream(ext, streams, blockIdx.y);
    out = of_stream(out, streams, blockIdx.y);
    const int p = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    float y[4];
    float sum = 0.f;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int c = tid + 256 * i;
        float r = b[c];
#pragma unroll
        for (int k = 0; k < 7; ++k) r = fmaf(w[c * 7 + k], ext[(size_t)(p + k) * 1024 + c], r);
        y[i] = r;
        sum += r;
    }
    sum = wave_sum(sum);
    if (lane == 0) red[wave] = sum;
    __syncthreads();
    const float mean = (red[0] + red[1] + red[2] + red[3]) / 1024.0f;
    __syncthreads();
    float var = 0.f;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const float c = y[i] - mean;
        var = fmaf(c, c, var);
    }
    var = wave_sum(var);
    if (lane == 0) red[wave] = var;
    __syncthreads();
    const float scale = 1.0f / sqrtf((red[0] + red[1] + red[2] + red[3]) / 1024.0f + 1.0e-6f);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int c = tid + 256 * i;
        out[(size_t)p * 1024 + c] = (y[i] - mean) * scale * ln_w[c] + ln_b[c];
    }
}

// ---------------------------------------------------------------------------
// Final causal convolution 96 -> 1 (CS:1699-1782 with the im2col column order
// channel-major, tap-minor), bias, clamp (CS:1126-1131), PCM (CS:1133-1143).
// ---------------------------------------------------------------------------
// Four lanes per position, each a sequential channel-major, tap-minor fmaf
// chain over 24 of the 96 channels (float4 reads), then the four partial sums
// added in channel-group order.
__global__ __launch_bounds__(256) void final_conv_pcm_kernel(const float* ext, int positions, const float* w,
                                                             const float* b, PcmTargets targets, float* preclamp,
                                                             float* clamped, Streams streams) {
    __shared__ float ws[96 * 7];
    ext = of_stream(ext, streams, blockIdx.y);
    preclamp = of_stream(preclamp, streams, blockIdx.y);
    clamped = of_stream(clamped, streams, blockIdx.y);
    int16_t* pcm = targets.pcm[blockIdx.y];
    for (int i = threadIdx.x; i < 96 * 7; i += 256) ws[i] = w[i];
    __syncthreads();
    const int lane = threadIdx.x & 63;
    const int group = lane >> 4;  // channels 24 * group .. + 23
    const int p = blockIdx.x * 64 + (threadIdx.x >> 6) * 16 + (lane & 15);
    const int pc = min(p, positions - 1);
    float4 x[7][6];
#pragma unroll
    for (int t = 0; t < 7; ++t)
#pragma unroll
        for (int q = 0; q < 6; ++q) x[t][q] = load4(ext + (size_t)(pc + t) * 96 + group * 24 + q * 4);
    float acc = 0.f;
#pragma unroll
    for (int q = 0; q < 6; ++q) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int c = group * 24 + q * 4 + e;
#pragma unroll
            for (int t = 0; t < 7; ++t) {
                const float xv = e == 0 ? x[t][q].x : e == 1 ? x[t][q].y : e == 2 ? x[t][q].z : x[t][q].w;
                acc = fmaf(xv, ws[c * 7 + t], acc);
            }
        }
    }
    // lanes r, r + 16, r + 32, r + 48 hold the four groups of position r
    const float g1 = __shfl(acc, (lane & 15) + 16, 64), g2 = __shfl(acc, (lane & 15) + 32, 64),
                g3 = __shfl(acc, (lane & 15) + 48, 64);
    if (group != 0 || p >= positions) return;
    const float v = ((acc + g1) + g2) + g3 + b[0];
    preclamp[p] = v;
    const float c = fminf(1.0f, fmaxf(-1.0f, v));
    clamped[p] = c;
    const float scaled = roundf(c * 32767.0f);
    pcm[p] = (int16_t)fminf(32767.0f, fmaxf(-32768.0f, scaled));
}

// ---------------------------------------------------------------------------
// Deterministic state-machine fixture (CS:185-318, 4518-4740): integer
// stand-ins for the pre-convolution (3x + 2 h1 - h2) / 4 over the weighted code
// sum, two repeats, four transposed-convolution overlaps (3x + previous) / 4
// with carried tails, and x * 8 saturated to 16 bits.  One block; the stages
// alternate between two LDS buffers.  state: [0..1] pre-conv history,
// [2..21] the tails of strides 8, 5, 4, 3.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void fixture_packet_kernel(const uint16_t* codes, int frames, int* state,
                                                             int16_t* pcm) {
    __shared__ int buf[2][kMaxFrames * kSamplesPerFrame];
    __shared__ int tails[20];
    const int tid = threadIdx.x;
    if (tid < 20) tails[tid] = state[2 + tid];
    if (tid == 0) {
        int h1 = state[0], h2 = state[1];
        for (int f = 0; f < frames; ++f) {
            int sum = 0;
            for (int cb = 0; cb < kCodebooks; ++cb) sum += (codes[f * kCodebooks + cb] & 2047) * (cb + 1);
            const int centered = (sum & 4095) - 2048;
            const int filtered = (3 * centered + 2 * h1 - h2) / 4;
            h2 = h1;
            h1 = centered;
            for (int r = 0; r < 4; ++r) buf[0][4 * f + r] = filtered;  // repeat x2, x2
        }
        state[0] = h1;
        state[1] = h2;
    }
    __syncthreads();
    int n = 4 * frames, src = 0, tail_base = 0;
    for (int stage = 0; stage < 4; ++stage) {
        const int stride = kStride[stage];
        const int* in = buf[src];
        int* out = buf[src ^ 1];
        for (int i = tid; i < n * stride; i += 256) {
            const int ip = i / stride, phase = i - ip * stride;
            const int previous = ip == 0 ? tails[tail_base + phase] : in[ip - 1];
            out[i] = (3 * in[ip] + previous) / 4;
        }
        __syncthreads();
        if (tid < stride) tails[tail_base + tid] = in[n - 1];
        __syncthreads();
        tail_base += stride;
        n *= stride;
        src ^= 1;
    }
    for (int i = tid; i < n; i += 256) {
        const int v = buf[src][i] * 8;
        pcm[i] = (int16_t)(v > 32767 ? 32767 : (v < -32768 ? -32768 : v));
    }
    if (tid < 20) state[2 + tid] = tails[tid];
}

// ---------------------------------------------------------------------------
// load-time kernels
// ---------------------------------------------------------------------------
__global__ void bf16_to_f32_kernel(const uint16_t* src, size_t count, float* dst) {
    for (size_t i = blockIdx.x * 256ull + threadIdx.x; i < count; i += (size_t)gridDim.x * 256)
        dst[i] = __uint_as_float((unsigned)src[i] << 16);
}

__global__ void repack_conv_kernel(const float* src, int out_ch, int in_ch, int taps, float* dst) {
    const size_t total = (size_t)out_ch * in_ch * taps;
    for (size_t i = blockIdx.x * 256ull + threadIdx.x; i < total; i += (size_t)gridDim.x * 256) {
        const size_t o = i / ((size_t)taps * in_ch);
        const size_t rem = i - o * taps * in_ch;
        const size_t t = rem / in_ch, c = rem - t * in_ch;
        dst[i] = src[(o * in_ch + c) * taps + t];
    }
}

__global__ void repack_transpose_kernel(const float* src, int in_ch, int out_ch, int stride, int overlap,
                                        float* dst) {
    const int span = overlap ? 2 * stride : stride;
    const int taps = overlap ? 2 : 1;
    const size_t k = (size_t)taps * in_ch;
    const size_t total = (size_t)stride * out_ch * k;
    for (size_t i = blockIdx.x * 256ull + threadIdx.x; i < total; i += (size_t)gridDim.x * 256) {
        const size_t row = i / k, col = i - row * k;
        const int phase = (int)(row / out_ch), o = (int)(row - (size_t)phase * out_ch);
        const int tap = (int)(col / in_ch), c = (int)(col - (size_t)tap * in_ch);
        const int kernel_index = overlap && tap == 0 ? stride + phase : phase;
        dst[i] = src[((size_t)c * out_ch + o) * span + kernel_index];
    }
}

__global__ void snake_params_kernel(float* alpha, float* beta, int channels) {
    const int c = blockIdx.x * 256 + threadIdx.x;
    if (c < channels) {
        alpha[c] = expf(alpha[c]);
        beta[c] = expf(beta[c]) + 1.0e-9f;
    }
}

__global__ void fill_f32_kernel(float* dst, size_t count, float value) {
    for (size_t i = blockIdx.x * 256ull + threadIdx.x; i < count; i += (size_t)gridDim.x * 256) dst[i] = value;
}

}  // namespace

// ---------------------------------------------------------------------------
// launchers
// ---------------------------------------------------------------------------
namespace {
bool valid(const Streams& s) { return s.count >= 1 && s.count <= kMaxStreams; }
}  // namespace

template <int kChunks, int kRows>
static void launch_rows_count(const RowsGemvArgs& g, hipStream_t stream) {
    const dim3 grid(g.n / kGemvWaves, g.streams.count);
    if (g.epilogue == kRowsSiluPair) rows_gemv_kernel<kChunks, kRows, true><<<grid, 64 * kGemvWaves, 0, stream>>>(g);
    else rows_gemv_kernel<kChunks, kRows, false><<<grid, 64 * kGemvWaves, 0, stream>>>(g);
}

template <int kChunks>
static void launch_rows_chunks(const RowsGemvArgs& g, hipStream_t stream) {
    if (g.rows == 1) launch_rows_count<kChunks, 1>(g, stream);
    else if (g.rows == 2) launch_rows_count<kChunks, 2>(g, stream);
    else launch_rows_count<kChunks, 4>(g, stream);
}

hipError_t launch_rows_gemv(const RowsGemvArgs& g, hipStream_t stream) {
    if (g.rows < 1 || g.rows > kMaxRows || g.k % 256 || g.ldx % 4 || g.n < kGemvWaves || g.n % kGemvWaves ||
        !valid(g.streams))
        return hipErrorInvalidValue;
    switch (g.k / 256) {
        case 2: launch_rows_chunks<2>(g, stream); break;
        case 4: launch_rows_chunks<4>(g, stream); break;
        case 6: launch_rows_chunks<6>(g, stream); break;
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

hipError_t launch_codec_attention(const float* qkv, int frames, const unsigned long long* position,
                                  const float* rotations, float* kv_k, float* kv_v, float* out, const Streams& streams,
                                  hipStream_t stream) {
    if (frames < 1 || frames > kMaxFrames || !valid(streams)) return hipErrorInvalidValue;
    codec_attention_kernel<<<dim3(kHeads, frames, streams.count), 256, 0, stream>>>(qkv, frames, position, rotations, kv_k,
                                                                                   kv_v, out, streams);
    return hipGetLastError();
}

hipError_t launch_codec_frontend(const uint16_t* codes, int frames, const float* const* embeddings,
                                 const float* const* usages, float* x, const unsigned long long* position,
                                 float* rotations, const CopySegment* seg, int segments, const Streams& streams,
                                 hipStream_t stream) {
    if (frames < 1 || frames > kMaxFrames || segments < 2 || !valid(streams)) return hipErrorInvalidValue;
    FrontendTables t;
    for (int i = 0; i < kCodebooks; ++i) {
        t.emb[i] = embeddings[i];
        t.usage[i] = usages[i];
    }
    codec_frontend_kernel<<<dim3(8, segments, streams.count), 256, 0, stream>>>(codes, frames, t, x, position, rotations,
                                                                               seg, streams);
    return hipGetLastError();
}

hipError_t launch_copy_segments(const CopySegment* seg, int segments, const Streams& streams, hipStream_t stream) {
    if (!valid(streams)) return hipErrorInvalidValue;
    if (segments <= 0) return hipSuccess;
    copy_segments_kernel<<<dim3(8, segments, streams.count), 256, 0, stream>>>(seg, streams);
    return hipGetLastError();
}

hipError_t launch_dwconv_layernorm(const float* ext, int positions, const float* w, const float* b,
                                   const float* ln_w, const float* ln_b, float* out, const Streams& streams,
                                   hipStream_t stream) {
    if (positions < 1 || !valid(streams)) return hipErrorInvalidValue;
    dwconv_layernorm_kernel<<<dim3(positions, streams.count), 256, 0, stream>>>(ext, w, b, ln_w, ln_b, out, streams);
    return hipGetLastError();
}

hipError_t launch_final_conv_pcm(const float* ext, int positions, const float* w, const float* b, const PcmTargets& pcm,
                                 float* preclamp, float* clamped, const Streams& streams, hipStream_t stream) {
    if (positions < 1 || !preclamp || !clamped || !valid(streams)) return hipErrorInvalidValue;
    final_conv_pcm_kernel<<<dim3((positions + 63) / 64, streams.count), 256, 0, stream>>>(ext, positions, w, b, pcm,
                                                                                         preclamp, clamped, streams);
    return hipGetLastError();
}

hipError_t launch_fixture_packet(const uint16_t* codes, int frames, int* state, int16_t* pcm, hipStream_t stream) {
    if (frames < 1 || frames > kMaxFrames) return hipErrorInvalidValue;
    fixture_packet_kernel<<<1, 256, 0, stream>>>(codes, frames, state, pcm);
    return hipGetLastError();
}

hipError_t launch_bf16_to_f32(const uint16_t* src, size_t count, float* dst, hipStream_t stream) {
    bf16_to_f32_kernel<<<blocks_for(count), 256, 0, stream>>>(src, count, dst);
    return hipGetLastError();
}

hipError_t launch_repack_conv(const float* src, int out_ch, int in_ch, int taps, float* dst, hipStream_t stream) {
    repack_conv_kernel<<<blocks_for((size_t)out_ch * in_ch * taps), 256, 0, stream>>>(src, out_ch, in_ch, taps, dst);
    return hipGetLastError();
}

hipError_t launch_repack_transpose(const float* src, int in_ch, int out_ch, int stride, bool overlap, float* dst,
                                   hipStream_t stream) {
    const size_t total = (size_t)stride * out_ch * in_ch * (overlap ? 2 : 1);
    repack_transpose_kernel<<<blocks_for(total), 256, 0, stream>>>(src, in_ch, out_ch, stride, overlap ? 1 : 0, dst);
    return hipGetLastError();
}

hipError_t launch_snake_params(float* alpha, float* beta, int channels, hipStream_t stream) {
    snake_params_kernel<<<(channels + 255) / 256, 256, 0, stream>>>(alpha, beta, channels);
    return hipGetLastError();
}

hipError_t launch_fill_f32(float* dst, size_t count, float value, hipStream_t stream) {
    fill_f32_kernel<<<blocks_for(count), 256, 0, stream>>>(dst, count, value);
    return hipGetLastError();
}

}  // namespace q3c
