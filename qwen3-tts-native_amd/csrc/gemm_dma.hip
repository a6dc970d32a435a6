// bf16 GEMM of the prompt prefill whose operands reach LDS by direct loads
// (global_load_lds, 16 bytes a lane):
//
//   C[m][n] = epilogue( sum_k A[m][k] * B[n][k] )      (fp32 accumulation)
//
// A block owns a kBM x kBN tile; K advances 64 at a time through kStages LDS
// buffers, the loads of the next kStages - 1 steps in flight while the waves
// (kWM x kWN, each a grid of v_mfma_f32_16x16x32_bf16 tiles) work on a step;
// one barrier a step.  An LDS row holds the step's 64 values of a matrix row
// as eight 16-byte chunks, chunk c at slot c ^ ((row >> 1) & 7): a direct load
// writes its 64 lanes' chunks side by side, so the swizzle is applied to the
// chunk that each lane reads from memory, and the 16 rows x 4 chunks of one
// fragment read fall into distinct banks without padding.  The buffers are
// separate __shared__ objects and the steps unrolled over them: the compiler
// then knows that a fragment read does not touch a buffer still being filled
// and adds no wait of its own for the loads.
//
// Bound: at 512 rows and up by LDS reads and the blocks' L2 reads (a 64 x 64
// tile reads 16 KB a step for 128 matrix-core cycles a wave), at short prompts
// by the weights' stream and the launch.  One talker layer's products (QKV, O,
// gate and up, down), register-staged tiles before -> here, us: 33 rows 70 ->
// 45, 512 rows 155 -> 92, 801 rows 232 -> 129.
//
// The product is formed transposed (B's rows as the MFMA's A operand), so a
// lane holds four consecutive columns of one row and stores 8 bytes.
#include <algorithm>

#include "head_device.hpp"
#include "q3_common.hpp"
#include "q3_math.h"

namespace q3 {
namespace {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float floatx4_t __attribute__((ext_vector_type(4)));
using lds_word = __attribute__((address_space(3))) unsigned int;
using global_word = const __attribute__((address_space(1))) unsigned int;

constexpr int kStep = 64;  // K per step

// s_waitcnt immediate: at most `vm` vector loads outstanding, no LDS operation
constexpr int wait_imm(int vm) { return (vm & 15) | ((vm >> 4) << 14) | (7 << 4); }

template <int kLoads>
__device__ __forceinline__ void wait_and_sync() {
    static_assert(kLoads < 64, "vmcnt");
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(wait_imm(kLoads));
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

// The text projection's products, which the decode step sums in fp32 by short
// chains and a tree: a step's 64 values are summed by the matrix cores from
// zero, the steps in double.  One chain over K is further from the exact sum
// (K 2048, int8 weights, rms error in 2^-24 of the sums' rms: 2.6 with one
// chain, 0.99 in the decode step's order), and a prompt's first layer then
// holds twice the values on the wrong side of a rounding step (1.05 %, 0.52 %
// in the decode step's order, 0.26 % here).  The conversions and additions hide
// behind the loads: prefills of 33 to 1024 rows are within 1 %.
constexpr bool is_wide(int epilogue) { return epilogue == kGemmScaleBias || epilogue == kGemmScaleBiasSilu; }

// A gate and an up product in one tile: C = silu_gate of their bf16 values.
constexpr int kGemmGated = 16;

// Four consecutive columns of one row.  Rounding as the separate launches':
// the product to bf16, then the residual add, silu_gate over the gate product
// in C, or the bias (with the text projection's scale and SiLU).
template <int kEpilogue>
__device__ __forceinline__ void store4(const Bf16GemmArgs& g, int row, int col, const floatx4_t& v) {
    bf16_t* out = g.c + static_cast<size_t>(row) * g.ldc + col;
    ushort4 r;
    if constexpr (kEpilogue == kGemmAddInto) {
        const ushort4 o = *reinterpret_cast<const ushort4*>(out);
        r.x = f2bf(bf2f(o.x) + round_bf(v[0]));
        r.y = f2bf(bf2f(o.y) + round_bf(v[1]));
        r.z = f2bf(bf2f(o.z) + round_bf(v[2]));
        r.w = f2bf(bf2f(o.w) + round_bf(v[3]));
    } else if constexpr (kEpilogue == kGemmSiluGateInto) {
        const ushort4 o = *reinterpret_cast<const ushort4*>(out);
        auto one = [](bf16_t gate, float up) {
            const float x = bf2f(gate);
            return f2bf(round_bf(x / (1.0f + q3_expf(-x))) * round_bf(up));
        };
        r.x = one(o.x, v[0]);
        r.y = one(o.y, v[1]);
        r.z = one(o.z, v[2]);
        r.w = one(o.w, v[3]);
    } else if constexpr (kEpilogue == kGemmScaleBias || kEpilogue == kGemmScaleBiasSilu) {
        const float4 s = *reinterpret_cast<const float4*>(g.scales + col);
        const ushort4 b = *reinterpret_cast<const ushort4*>(g.bias + col);
        auto one = [](float x, bf16_t bias) {
            float y = round_bf(x) + bf2f(bias);
            if constexpr (kEpilogue == kGemmScaleBiasSilu) y *= 1.0f / (1.0f + q3_expf(-y));
            return f2bf(y);
        };
        r.x = one(v[0] * s.x, b.x);
        r.y = one(v[1] * s.y, b.y);
        r.z = one(v[2] * s.z, b.z);
        r.w = one(v[3] * s.w, b.w);
    } else {
        r.x = f2bf(v[0]);
        r.y = f2bf(v[1]);
        r.z = f2bf(v[2]);
        r.w = f2bf(v[3]);
    }
    *reinterpret_cast<ushort4*>(out) = r;
}

__device__ __forceinline__ void store_gated4(const Bf16GemmArgs& g, int row, int col, const floatx4_t& gate,
                                             const floatx4_t& up) {
    auto one = [](float a, float b) {
        const float x = round_bf(a);
        return f2bf(round_bf(x / (1.0f + q3_expf(-x))) * round_bf(b));
    };
    ushort4 r;
    r.x = one(gate[0], up[0]);
    r.y = one(gate[1], up[1]);
    r.z = one(gate[2], up[2]);
    r.w = one(gate[3], up[3]);
    *reinterpret_cast<ushort4*>(g.c + static_cast<size_t>(row) * g.ldc + col) = r;
}

// Grid: blocks of one column panel (all row tiles of a B panel) have numbers
// 8 apart, so they run on one XCD and read the panel through its L2 once:
// block -> xcd = block % 8, i = block / 8, panel = xcd + 8 * (i / row tiles),
// row tile = i % row tiles; grid.y = K slice.
// kGated: the tile's columns are kBN / 2 gate columns (rows of b) and the
// same kBN / 2 up columns (rows of b2), and C has n = the up columns.
template <int kBM, int kBN, int kWM, int kWN, int kStages, int kEpilogue>
__global__ __launch_bounds__(64 * kWM * kWN) void gemm_dma_kernel(Bf16GemmArgs g, int row_tiles, int panels,
                                                                   int steps_per_split) {
    constexpr bool kGated = kEpilogue == kGemmGated;
    constexpr bool kWide = is_wide(kEpilogue);
    constexpr int kWaves = kWM * kWN;
    constexpr int kTM = kBM / 16 / kWM, kTN = kBN / 16 / kWN;
    constexpr int kLoads = (kBM + kBN) / 8 / kWaves;  // loads a wave issues per step, 8 rows each
    static_assert(kBM % (16 * kWM) == 0 && kBN % (16 * kWN) == 0 && (kBM + kBN) % (8 * kWaves) == 0, "tile");
    static_assert(kStages >= 2 && kStages <= 4, "stages");
    static_assert(!kGated || kTN % 2 == 0, "gate and up tiles in pairs");
    constexpr int kStageElements = (kBM + kBN) * kStep;
    __shared__ __align__(16) bf16_t buffer0[kStageElements];
    __shared__ __align__(16) bf16_t buffer1[kStageElements];
    __shared__ __align__(16) bf16_t buffer2[kStages > 2 ? kStageElements : 8];
    __shared__ __align__(16) bf16_t buffer3[kStages > 3 ? kStageElements : 8];

    const int xcd = blockIdx.x & 7, index = blockIdx.x >> 3;
    const int panel = xcd + 8 * (index / row_tiles);
    if (panel >= panels) return;  // the whole block
    const int m0 = (index % row_tiles) * kBM;
    constexpr int kColumns = kGated ? kBN / 2 : kBN;
    const int n0 = panel * kColumns;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int first = blockIdx.y * steps_per_split;
    const int steps = min(g.k / kStep - first, steps_per_split);

    // this lane's source of load i: chunk (slot ^ swizzle) of tile row
    // 8 * (wave + kWaves * i) + lane / 8; rows past a matrix repeat its last
    // row (their products are never stored)
    const bf16_t* source[kLoads];
#pragma unroll
    for (int i = 0; i < kLoads; ++i) {
        const int row = 8 * (wave + kWaves * i) + (lane >> 3);
        const int chunk = (lane & 7) ^ ((row >> 1) & 7);
        const bf16_t* base;
        if (row < kBM) {
            base = g.a + static_cast<size_t>(min(m0 + row, g.m - 1)) * g.lda;
        } else if (kGated) {
            const int column = row - kBM;
            const bool up = column >= kColumns;
            base = (up ? g.b2 : g.b) + static_cast<size_t>(min(n0 + column - (up ? kColumns : 0), g.n - 1)) * g.ldb;
        } else {
            const int column = min(n0 + row - kBM, g.n - 1);
            base = g.b + static_cast<size_t>(column) * g.ldb;
            if (g.b2 != nullptr && column >= g.b2_row) base = g.b2 + static_cast<size_t>(column - g.b2_row) * g.ldb;
            if (g.b3 != nullptr && column >= g.b3_row) base = g.b3 + static_cast<size_t>(column - g.b3_row) * g.ldb;
        }
        source[i] = base + static_cast<size_t>(first) * kStep + chunk * 8;
    }
    auto buffer = [&](int stage) -> bf16_t* {
        return stage == 0 ? buffer0 : stage == 1 ? buffer1 : stage == 2 ? buffer2 : buffer3;
    };
    auto load = [&](int stage) {  // the next step into `stage`
        bf16_t* to = buffer(stage);
#pragma unroll
        for (int i = 0; i < kLoads; ++i) {
            __builtin_amdgcn_global_load_lds((global_word*)source[i], (lds_word*)(to + (wave + kWaves * i) * 512), 16, 0, 0);
            source[i] += kStep;
        }
    };

    const int wm = (wave / kWN) * (16 * kTM), wn = wave % kWN;
    const int m = lane & 15, group = lane >> 4;
    // tile column of the wave's j-th 16 columns (LDS row kBM + column)
    auto column_of = [&](int j) {
        if (kGated) return (j < kTN / 2 ? 0 : kColumns) + (wn * (kTN / 2) + j % (kTN / 2)) * 16;
        return (wn * kTN + j) * 16;
    };
    floatx4_t acc[kTM][kTN];
    double wide[kWide ? kTM : 1][kWide ? kTN : 1][4];
#pragma unroll
    for (int i = 0; i < kTM; ++i)
#pragma unroll
        for (int j = 0; j < kTN; ++j) acc[i][j] = floatx4_t{0.f, 0.f, 0.f, 0.f};
    if constexpr (kWide) {
#pragma unroll
        for (int i = 0; i < kTM; ++i)
#pragma unroll
            for (int j = 0; j < kTN; ++j)
#pragma unroll
                for (int r = 0; r < 4; ++r) wide[i][j][r] = 0.0;
    }
    // lane offsets of the fragments of the step's two halves; the rest of an
    // address is a constant
    const int slot0 = (group ^ (m >> 1)) * 8, slot1 = slot0 ^ 32;
    const int a_lane = (wm + m) * kStep, b_lane = (kBM + column_of(0) + m) * kStep;
    auto compute = [&](int stage) {
        const bf16_t* from = buffer(stage);
#pragma unroll
        for (int kk = 0; kk < 2; ++kk) {
            const bf16_t* a_from = from + (a_lane + (kk == 0 ? slot0 : slot1));
            const bf16_t* b_from = from + (b_lane + (kk == 0 ? slot0 : slot1));
            bf16x8_t af[kTM], bf[kTN];
#pragma unroll
            for (int i = 0; i < kTM; ++i) af[i] = *reinterpret_cast<const bf16x8_t*>(a_from + 16 * i * kStep);
#pragma unroll
            for (int j = 0; j < kTN; ++j) {
                const int column = kGated ? (j < kTN / 2 ? 0 : kColumns) + 16 * (j % (kTN / 2)) : 16 * j;
                bf[j] = *reinterpret_cast<const bf16x8_t*>(b_from + column * kStep);
            }
#pragma unroll
            for (int i = 0; i < kTM; ++i)
#pragma unroll
                for (int j = 0; j < kTN; ++j) {
                    const floatx4_t onto = kWide && kk == 0 ? floatx4_t{0.f, 0.f, 0.f, 0.f} : acc[i][j];
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bf[j], af[i], onto, 0, 0, 0);
                }
        }
        if constexpr (kWide) {
#pragma unroll
            for (int i = 0; i < kTM; ++i)
#pragma unroll
                for (int j = 0; j < kTN; ++j)
#pragma unroll
                    for (int r = 0; r < 4; ++r) wide[i][j][r] += static_cast<double>(acc[i][j][r]);
        }
    };

    // Steps 0 .. kStages - 2 requested; then, per step: wait until only the
    // later steps' loads are outstanding, synchronize (the step is complete
    // for every wave, and the buffer of the step before is free), request
    // step + kStages - 1 into that buffer, compute.  The last kStages - 1
    // steps wait once for everything.
#pragma unroll
    for (int s = 0; s < kStages - 1; ++s)
        if (s < steps) load(s);
    const int pipelined = steps - (kStages - 1);
    int done = 0;
    bool more = true;
    while (more) {
#pragma unroll
        for (int stage = 0; stage < kStages; ++stage) {
            if (!more) break;
            if (done >= pipelined) {
                wait_and_sync<0>();
#pragma unroll
                for (int t = 0; t < kStages - 1; ++t)
                    if (done + t < steps) compute((stage + t) % kStages);
                more = false;
                break;
            }
            wait_and_sync<(kStages - 2) * kLoads>();
            load((stage + kStages - 1) % kStages);
            compute(stage);
            ++done;
        }
    }

    if constexpr (kWide) {
#pragma unroll
        for (int i = 0; i < kTM; ++i)
#pragma unroll
            for (int j = 0; j < kTN; ++j)
#pragma unroll
                for (int r = 0; r < 4; ++r) acc[i][j][r] = static_cast<float>(wide[i][j][r]);
    }
    // acc[i][j][r] = C[m0 + wm + 16 i + m][column + 4 group + r]
    const bool split = gridDim.y > 1;
    float* partial = split ? g.partial + static_cast<size_t>(blockIdx.y) * g.m * g.n : nullptr;
#pragma unroll
    for (int i = 0; i < kTM; ++i) {
        const int row = m0 + wm + 16 * i + m;
        if (row >= g.m) continue;
        if constexpr (kGated) {
#pragma unroll
            for (int j = 0; j < kTN / 2; ++j) {
                const int col = n0 + column_of(j) + 4 * group;
                if (col < g.n) store_gated4(g, row, col, acc[i][j], acc[i][j + kTN / 2]);
            }
        } else {
#pragma unroll
            for (int j = 0; j < kTN; ++j) {
                const int col = n0 + column_of(j) + 4 * group;
                if (col >= g.n) continue;
                if (split) *reinterpret_cast<floatx4_t*>(partial + static_cast<size_t>(row) * g.n + col) = acc[i][j];
                else store4<kEpilogue>(g, row, col, acc[i][j]);
            }
        }
    }
}

// The (at most 8) slices' sums, added in slice order; four columns a thread.
template <int kEpilogue>
__global__ __launch_bounds__(256) void gemm_dma_reduce_kernel(Bf16GemmArgs g, int splits) {
    const int quads = g.n / 4;
    const int t = blockIdx.x * 256 + threadIdx.x;
    if (t >= quads * g.m) return;
    const int row = t / quads, col = (t - row * quads) * 4;
    const size_t slice = static_cast<size_t>(g.m) * g.n;
    const float* p = g.partial + static_cast<size_t>(row) * g.n + col;
    floatx4_t v[8];
#pragma unroll
    for (int s = 0; s < 8; ++s)
        if (s < splits) v[s] = *reinterpret_cast<const floatx4_t*>(p + s * slice);
    floatx4_t sum = v[0];
    if constexpr (is_wide(kEpilogue)) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            double total = v[0][r];
#pragma unroll
            for (int s = 1; s < 8; ++s)
                if (s < splits) total += static_cast<double>(v[s][r]);
            sum[r] = static_cast<float>(total);
        }
    } else {
#pragma unroll
        for (int s = 1; s < 8; ++s)
            if (s < splits) sum += v[s];
    }
    store4<kEpilogue>(g, row, col, sum);
}

// The same with the RMSNorm that follows (rms_norm_rows' arithmetic and order,
// so its bits): a block per row keeps the finished row in LDS, which saves the
// norm's launch and its read of the row.  With the residual add: 33 rows 3.8 +
// 3.2 us as two launches, 4.3 us here.
constexpr int kNormColumns = 2048;  // a thread's two quads of columns
__global__ __launch_bounds__(256) void gemm_dma_reduce_norm_kernel(Bf16GemmArgs g, int splits) {
    __shared__ __align__(16) bf16_t row_lds[kNormColumns];
    __shared__ float partial_lds[256];
    const int row = blockIdx.x, tid = threadIdx.x;
    const size_t slice = static_cast<size_t>(g.m) * g.n;
    bf16_t* out = g.c + static_cast<size_t>(row) * g.ldc;
    // everything this thread reads, requested together
    floatx4_t v[2][8];
    ushort4 residual[2], gain[2];
#pragma unroll
    for (int q = 0; q < 2; ++q) {
        const int col = min(tid * 4 + 1024 * q, g.n - 4);
        const float* p = g.partial + static_cast<size_t>(row) * g.n + col;
#pragma unroll
        for (int s = 0; s < 8; ++s)
            if (s < splits) v[q][s] = *reinterpret_cast<const floatx4_t*>(p + s * slice);
        residual[q] = *reinterpret_cast<const ushort4*>(out + col);
        gain[q] = *reinterpret_cast<const ushort4*>(g.norm_weight + col);
    }
#pragma unroll
    for (int q = 0; q < 2; ++q) {
        const int col = tid * 4 + 1024 * q;
        if (col >= g.n) continue;
        floatx4_t sum = v[q][0];
#pragma unroll
        for (int s = 1; s < 8; ++s)
            if (s < splits) sum += v[q][s];
        ushort4 r;
        r.x = f2bf(bf2f(residual[q].x) + round_bf(sum[0]));
        r.y = f2bf(bf2f(residual[q].y) + round_bf(sum[1]));
        r.z = f2bf(bf2f(residual[q].z) + round_bf(sum[2]));
        r.w = f2bf(bf2f(residual[q].w) + round_bf(sum[3]));
        *reinterpret_cast<ushort4*>(out + col) = r;
        *reinterpret_cast<ushort4*>(&row_lds[col]) = r;
    }
    __syncthreads();
    float square = 0.f;
#pragma unroll
    for (int i = 0; i < kNormColumns / 256; ++i) {
        if (tid + 256 * i < g.n) {
            const float x = bf2f(row_lds[tid + 256 * i]);
            square = fmaf(x, x, square);
        }
    }
    partial_lds[tid] = square;
    __syncthreads();
    const int lane = tid & 63;
    const float total = head_detail::wave_tree256(partial_lds[lane], partial_lds[lane + 64], partial_lds[lane + 128],
                                                  partial_lds[lane + 192]);
    const float inverse = 1.0f / sqrtf(total / static_cast<float>(g.n) + g.norm_epsilon);
#pragma unroll
    for (int q = 0; q < 2; ++q) {
        const int col = tid * 4 + 1024 * q;
        if (col >= g.n) continue;
        const ushort4 x = *reinterpret_cast<const ushort4*>(&row_lds[col]);
        ushort4 o;
        o.x = f2bf(round_bf(bf2f(x.x) * inverse) * bf2f(gain[q].x));
        o.y = f2bf(round_bf(bf2f(x.y) * inverse) * bf2f(gain[q].y));
        o.z = f2bf(round_bf(bf2f(x.z) * inverse) * bf2f(gain[q].z));
        o.w = f2bf(round_bf(bf2f(x.w) * inverse) * bf2f(gain[q].w));
        *reinterpret_cast<ushort4*>(g.norm_out + static_cast<size_t>(row) * g.n + col) = o;
    }
}

template <int kBM, int kBN, int kWM, int kWN, int kStages, int kEpilogue>
hipError_t launch_tile(const Bf16GemmArgs& g, int splits, hipStream_t stream) {
    const int columns = kEpilogue == kGemmGated ? kBN / 2 : kBN;
    const int row_tiles = (g.m + kBM - 1) / kBM, panels = (g.n + columns - 1) / columns;
    const int steps = g.k / kStep;
    const int per = (steps + splits - 1) / splits;
    const int slices = (steps + per - 1) / per;  // no empty slice
    const dim3 grid((panels + 7) / 8 * 8 * row_tiles, slices);
    gemm_dma_kernel<kBM, kBN, kWM, kWN, kStages, kEpilogue><<<grid, 64 * kWM * kWN, 0, stream>>>(g, row_tiles, panels, per);
    hipError_t st = hipGetLastError();
    const bool norm = kEpilogue == kGemmAddInto && g.norm_out != nullptr;
    if (kEpilogue == kGemmStore && g.open_slices != nullptr && slices > 1) {  // the consumer adds them
        if (st == hipSuccess) *g.open_slices = slices;
        return st;
    }
    if constexpr (kEpilogue == kGemmAddInto) {
        if (st == hipSuccess && norm && slices > 1 && slices <= 8 && g.n <= kNormColumns) {
            gemm_dma_reduce_norm_kernel<<<g.m, 256, 0, stream>>>(g, slices);
            return hipGetLastError();
        }
    }
    if (st == hipSuccess && slices > 1) {
        gemm_dma_reduce_kernel<kEpilogue><<<(g.m * (g.n / 4) + 255) / 256, 256, 0, stream>>>(g, slices);
        st = hipGetLastError();
    }
    if (st == hipSuccess && norm)
        st = launch_rms_norm_rows(g.c, g.norm_weight, g.norm_out, g.m, g.n, g.norm_epsilon, stream);
    return st;
}

template <int kEpilogue>
hipError_t launch_plain(const Bf16GemmArgs& g, hipStream_t stream) {
    // Measured over N 2048 / 4096 at K 2048 and N 2048 at K 6144, 16..801
    // rows, weights from HBM (us; the K-sliced times hold the reduction):
    //  - deep products (K >= 4096) slice K, at least 12 steps a slice: 128 x
    //    128 tiles from 160 rows on (512 rows: 26.0 in 4 slices; 64 x 64 30+,
    //    128 x 64 in 2 28.5), 64 x 64 below (33 rows in 8 slices: 12.7; 64 x
    //    32 12.8, 16-row tiles 14+);
    //  - otherwise 128 x 128 once it fills three CUs in four unsliced (801 x
    //    4096: 21.7 against 25.2 for 128 x 64), 64 x 64 while that fills as
    //    many (512 x 2048: 13.3; 128 x 64 17+), 32 x 64 else (256 x 2048:
    //    10.9 against 12+), each row beyond 128;
    //  - up to 128 rows 64 x 32 (or the 32- and 16-row tile that holds them)
    //    in up to 4 slices (64 x 4096: 10.5; unsliced 12+).
    const int steps = g.k / kStep;
    auto tiles = [&](int bm, int bn) { return ((g.m + bm - 1) / bm) * ((g.n + bn - 1) / bn); };
    const size_t plane = static_cast<size_t>(g.m) * g.n;
    const int room = g.partial == nullptr ? 1 : static_cast<int>(std::min<size_t>(8, std::max<size_t>(1, g.partial_floats / plane)));
    if (g.k >= 4096) {
        const int most = std::min(room, steps / 12);
        if (g.m >= 160) {
            const int splits = std::max(1, std::min(most, 256 / tiles(128, 128)));
            return launch_tile<128, 128, 2, 4, 3, kEpilogue>(g, splits, stream);
        }
        auto splits = [&](int t) { return g.m > 128 ? most : std::max(1, std::min(most, (512 + t - 1) / t)); };
        if (g.m > 32) return launch_tile<64, 64, 2, 2, 3, kEpilogue>(g, splits(tiles(64, 64)), stream);
        if (g.m > 16) return launch_tile<32, 32, 1, 2, 4, kEpilogue>(g, splits(tiles(32, 32)), stream);
        return launch_tile<16, 32, 1, 2, 4, kEpilogue>(g, splits(tiles(16, 32)), stream);
    }
    if (g.m > 128 && g.norm_out != nullptr && g.n <= kNormColumns && room >= 2) {
        // two slices, whose reduction is then the norm's launch too (2048 x
        // 2048 and its norm: 512 rows 13.3 + 6 -> 16 us, 801 rows 15.7 + 6 ->
        // 19 us)
        if (tiles(64, 64) < 400) return launch_tile<64, 64, 2, 2, 3, kEpilogue>(g, 2, stream);
        return launch_tile<128, 128, 2, 4, 3, kEpilogue>(g, 2, stream);
    }
    if (g.m > 128) {
        if (tiles(128, 128) >= 192) return launch_tile<128, 128, 2, 4, 3, kEpilogue>(g, 1, stream);
        if (tiles(64, 64) >= 192) return launch_tile<64, 64, 2, 2, 3, kEpilogue>(g, 1, stream);
        return launch_tile<32, 64, 1, 4, 4, kEpilogue>(g, 1, stream);
    }
    const int most = std::min(std::min(room, 4), std::max(1, steps / 8));
    auto splits = [&](int t) { return std::max(1, std::min(most, (400 + t - 1) / t)); };
    if (g.m > 32) return launch_tile<64, 32, 2, 2, 4, kEpilogue>(g, splits(tiles(64, 32)), stream);
    if (g.m > 16) return launch_tile<32, 32, 1, 2, 4, kEpilogue>(g, splits(tiles(32, 32)), stream);
    return launch_tile<16, 32, 1, 2, 4, kEpilogue>(g, splits(tiles(16, 32)), stream);
}

hipError_t launch_gated(const Bf16GemmArgs& g, hipStream_t stream) {
    // Up to 128 rows the weights' stream counts: 32 gate and 32 up columns a
    // block (6144 + 6144 columns, K 2048, random weights from memory: 33 rows
    // 17.0 us, 64 rows 17.9 us, 2.8 TB/s; 64 x 128 20.6 and 21.3).
    if (g.m <= 16) return launch_tile<16, 64, 1, 2, 4, kGemmGated>(g, 1, stream);
    if (g.m <= 128) return launch_tile<64, 64, 2, 2, 4, kGemmGated>(g, 1, stream);
    // Beyond: the tile whose rounds over the 256 CUs cost least, as a launch
    // plus a time a round, fitted to all five over 129 to 1152 rows in one run
    // (us, K 2048, random weights from memory; a larger tile reads less and
    // rounds up more): 150 rows 24.5 with 96 x 128, 256 26.9 with 128 x 128,
    // 384 29.8 with 96 x 192, 512 34.8 with 128 x 192 (64 x 128 44.6), 801
    // 64.8 with 128 x 192 (two rounds; 64 x 128 in five 65.7, 96 x 192 75.8).
    // The pick is within 1 % of the best up to 1152 rows, 7 % beyond.
    struct Tile {
        int rows, columns;
        float launch, round;
    };
    const Tile tile[5] = {{128, 96, 3.0f, 31.0f}, {96, 96, 3.5f, 25.7f}, {128, 64, 4.0f, 22.0f}, {96, 64, 6.0f, 19.5f},
                          {64, 64, 6.5f, 11.8f}};
    int best = 0;
    float least = 0.f;
    for (int i = 0; i < 5; ++i) {
        const int blocks = ((g.m + tile[i].rows - 1) / tile[i].rows) * ((g.n + tile[i].columns - 1) / tile[i].columns);
        const float cost = tile[i].launch + static_cast<float>((blocks + 255) / 256) * tile[i].round;
        if (i == 0 || cost < least) {
            best = i;
            least = cost;
        }
    }
    switch (best) {
        case 0: return launch_tile<128, 192, 2, 2, 3, kGemmGated>(g, 1, stream);
        case 1: return launch_tile<96, 192, 2, 2, 3, kGemmGated>(g, 1, stream);
        case 2: return launch_tile<128, 128, 2, 2, 3, kGemmGated>(g, 1, stream);
        case 3: return launch_tile<96, 128, 2, 2, 4, kGemmGated>(g, 1, stream);
        default: return launch_tile<64, 128, 2, 2, 3, kGemmGated>(g, 1, stream);
    }
}

bool aligned(const void* p, unsigned bytes) { return (reinterpret_cast<uintptr_t>(p) & (bytes - 1)) == 0; }

}  // namespace

// What the direct loads and the 8-byte stores need; everything else runs
// gemm_bf16_kernel.
bool gemm_dma_takes(const Bf16GemmArgs& g) {
    if (g.force_tile != 0 || g.force_k_step != 0 || g.force_splits != 0 || g.batch != 1) return false;
    if (g.m <= 0 || g.n <= 0 || g.k <= 0 || g.k % kStep != 0 || g.n % 4 != 0 || g.ldc % 4 != 0 || g.lda % 8 != 0 ||
        g.ldb % 8 != 0 || g.lda < g.k || g.ldb < g.k || g.ldc < g.n) {
        return false;
    }
    if (!aligned(g.a, 16) || !aligned(g.b, 16) || !aligned(g.b2, 16) || !aligned(g.b3, 16) || !aligned(g.c, 8)) return false;
    if (g.partial != nullptr && !aligned(g.partial, 16)) return false;
    if (static_cast<long long>(g.m) * g.n > (1LL << 31) - 1) return false;
    if (g.norm_out != nullptr &&
        (g.epilogue != kGemmAddInto || g.norm_weight == nullptr || g.ldc != g.n ||
         !aligned(g.norm_out, 16) || !aligned(g.norm_weight, 16) || !aligned(g.c, 16) || g.n % 8 != 0)) {
        return false;
    }
    const bool biased = g.epilogue == kGemmScaleBias || g.epilogue == kGemmScaleBiasSilu;
    return !biased || (g.scales != nullptr && g.bias != nullptr && aligned(g.scales, 16) && aligned(g.bias, 8));
}

hipError_t launch_gemm_dma(const Bf16GemmArgs& g, hipStream_t stream) {
    if (g.a == nullptr || g.b == nullptr || g.c == nullptr || !gemm_dma_takes(g)) return hipErrorInvalidValue;
    switch (g.epilogue) {
        case kGemmStore: return launch_plain<kGemmStore>(g, stream);
        case kGemmAddInto: return launch_plain<kGemmAddInto>(g, stream);
        case kGemmSiluGateInto: return launch_plain<kGemmSiluGateInto>(g, stream);
        case kGemmScaleBias: return launch_plain<kGemmScaleBias>(g, stream);
        case kGemmScaleBiasSilu: return launch_plain<kGemmScaleBiasSilu>(g, stream);
        default: return hipErrorInvalidValue;
    }
}

hipError_t launch_gate_up_gemm(const Bf16GemmArgs& g, hipStream_t stream) {
    if (g.a == nullptr || g.b == nullptr || g.b2 == nullptr || g.c == nullptr || g.b3 != nullptr || !gemm_dma_takes(g))
        return hipErrorInvalidValue;
    return launch_gated(g, stream);
}

}  // namespace q3
