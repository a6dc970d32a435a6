// The decoder's products, out[p][col] = epilogue( sum_k A[p][k] * W[col][k] )
// in fp32 on the matrix cores (v_mfma_f32_16x16x4_f32), A read in place from
// an extended (history + packet) buffer: tap t of row p is buffer row
// p + t * dilation.  Two kernels:
//
//  - rows_kernel for up to 32 rows of K <= 1536 (the latent stages, a single
//    frame's first units): a block owns 16 columns, its waves take the 32-wide K
//    steps in turn straight from memory into the matrix operands' registers
//    (every weight is used by one wave only, so LDS would add nothing), and
//    their partial tiles meet in LDS.  Bound by the weights' stream and one
//    round of latency (1024 x 4096: 7.3 us, K slices and reduction before 10.9).
//  - tile_kernel for longer sequences: kBM x kBN tiles, operands through a
//    ring of direct-to-LDS loads, optionally kWK wave groups that each take
//    their own 32 of every 32 * kWK values of K (more waves a CU, and no
//    partial sums through memory).
//
// In both, element (p, col) is a sum over K in an order that depends on the
// layer and the packet's frames only, never on how many streams share the
// launch: a batch gives each stream the bits that it gets alone.
//
// Rows of several streams: row r of the launch is row r % m of stream r / m.
#include "codec.hpp"

#include <algorithm>

namespace q3c {

namespace {

typedef float floatx4 __attribute__((ext_vector_type(4)));
using lds_word = __attribute__((address_space(3))) unsigned int;
using global_word = const __attribute__((address_space(1))) unsigned int;

__device__ __forceinline__ floatx4 load4(const float* p) { return *reinterpret_cast<const floatx4*>(p); }

// (stream offset in floats, row within the stream) of launch row r
struct Row {
    ptrdiff_t delta;
    int p;
};
__device__ __forceinline__ Row locate(const ConvArgs& g, int r) {
    if (g.streams.count == 1) return {0, r};
    const int s = r / g.m;
    return {g.streams.delta[s] / static_cast<ptrdiff_t>(sizeof(float)), r - s * g.m};
}

// Four consecutive columns: bias (CS:407-412), GELU (CS:860-866), the scaled
// residual of ConvNeXt (gamma, CS:1432-1667) and of the transformer (layer
// scale), the residual unit's add (CS:1115-1124), then SnakeBeta (CS:882-898)
// into the next layer's input.
struct EpilogueIn {
    floatx4 bias, gamma, alpha, beta, residual;
};
__device__ __forceinline__ EpilogueIn load_epilogue(const ConvArgs& g, const Row& row, int col, int ch) {
    const floatx4 zero = {0.f, 0.f, 0.f, 0.f};
    EpilogueIn e;
    e.bias = g.bias ? load4(g.bias + ch) : zero;
    e.gamma = g.epilogue == kEpGammaResidual ? load4(g.gamma + ch) : zero;
    e.alpha = g.snake_out ? load4(g.snake_alpha + ch) : zero;
    e.beta = g.snake_out ? load4(g.snake_beta_den + ch) : zero;
    e.residual = g.epilogue == kEpGammaResidual || g.epilogue == kEpResidual
                     ? load4(g.residual + row.delta + static_cast<size_t>(row.p) * g.n + col)
                     : zero;
    return e;
}
__device__ __forceinline__ void store_epilogue(const ConvArgs& g, const Row& row, int col, const EpilogueIn& e, floatx4 v) {
    v += e.bias;
    if (g.epilogue == kEpGelu) {
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = 0.5f * v[i] * (1.0f + erff(v[i] * 0.7071067811865475f));
    } else if (g.epilogue == kEpGammaResidual) {
        v = e.residual + v * e.gamma;
    } else if (g.epilogue == kEpResidual) {
        v = v + e.residual;
    }
    const ptrdiff_t at = row.delta + static_cast<ptrdiff_t>(row.p) * g.n + col;
    if (g.out) *reinterpret_cast<floatx4*>(g.out + at) = v;
    if (g.snake_out) {
        floatx4 s;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const float x = sinf(v[i] * e.alpha[i]);
            s[i] = v[i] + (x * x) / e.beta[i];
        }
        *reinterpret_cast<floatx4*>(g.snake_out + at) = s;
    }
}

// ---------------------------------------------------------------------------
// Few rows.  kTM tiles of 16 rows a block; wave w of kWaves takes K steps w,
// w + kWaves, ...  Lane (m = lane & 15, group = lane >> 4) reads 8 consecutive
// floats at k = 8 group of weight row m and of activation row m of a step;
// MFMA e takes element e of both, so its four k slots are 8 g + e.
// ---------------------------------------------------------------------------
template <int kTM, int kWaves>
__global__ __launch_bounds__(64 * kWaves) void rows_kernel(ConvArgs g) {
    static_assert(kTM <= kWaves, "one output a thread");
    constexpr int kUnroll = kTM > 2 ? 2 : 4;  // steps whose loads are in flight together
    __shared__ __align__(16) float tiles[kWaves][kTM][4][17 * 4];  // [group][row] float4, padded
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int m = lane & 15, group = lane >> 4;
    const int col0 = blockIdx.x * 16;
    const int rows = g.m * g.streams.count;
    const int r0 = blockIdx.y * 16 * kTM;

    const float* w = g.w + static_cast<size_t>(col0 + m) * g.k + 8 * group;
    const float* x[kTM];
#pragma unroll
    for (int i = 0; i < kTM; ++i) {
        const Row row = locate(g, min(r0 + 16 * i + m, rows - 1));
        x[i] = g.a + row.delta + static_cast<size_t>(row.p) * g.channels_in + 8 * group;
    }
    // After the reduction thread t < 64 kTM finishes tile t / 64, row
    // (t / 4) % 16, columns 4 (t & 3) .. + 3; its operands are requested here,
    // beside the weights.
    const bool finishes = tid < kTM * 64;
    const int out_tile = tid >> 6, out_row = (tid >> 2) & 15, quad = tid & 3;
    const int out_r = min(r0 + 16 * out_tile + out_row, rows - 1), col = col0 + 4 * quad;
    const Row at_out = locate(g, out_r);
    EpilogueIn ein;
    if (finishes) ein = load_epilogue(g, at_out, col, col % g.channels_out);
    floatx4 acc[kTM];
#pragma unroll
    for (int i = 0; i < kTM; ++i) acc[i] = floatx4{0.f, 0.f, 0.f, 0.f};
    const int steps = g.k >> 5;
    // (tap, channel) of this wave's next step
    int tap = (32 * wave) / g.channels_in, chan = 32 * wave - tap * g.channels_in;
    const ptrdiff_t tap_stride = static_cast<ptrdiff_t>(g.dilation) * g.channels_in;
    for (int s0 = wave; s0 < steps; s0 += kWaves * kUnroll) {
        floatx4 wv[kUnroll][2], xv[kUnroll][kTM][2];
#pragma unroll
        for (int u = 0; u < kUnroll; ++u) {
            const int s = s0 + u * kWaves;
            if (s < steps) {
                wv[u][0] = load4(w + 32 * s);
                wv[u][1] = load4(w + 32 * s + 4);
                const ptrdiff_t at = tap * tap_stride + chan;
#pragma unroll
                for (int i = 0; i < kTM; ++i) {
                    xv[u][i][0] = load4(x[i] + at);
                    xv[u][i][1] = load4(x[i] + at + 4);
                }
                chan += 32 * kWaves;
                while (chan >= g.channels_in) chan -= g.channels_in, ++tap;
            }
        }
#pragma unroll
        for (int u = 0; u < kUnroll; ++u) {
            if (s0 + u * kWaves >= steps) break;
#pragma unroll
            for (int e = 0; e < 8; ++e)
#pragma unroll
                for (int i = 0; i < kTM; ++i)
                    acc[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(wv[u][e >> 2][e & 3], xv[u][i][e >> 2][e & 3], acc[i], 0, 0, 0);
        }
    }
    // acc[i] of lane (group, m): columns 4 group .. + 3 of row m
#pragma unroll
    for (int i = 0; i < kTM; ++i) *reinterpret_cast<floatx4*>(&tiles[wave][i][group][m * 4]) = acc[i];
    __syncthreads();
    if (!finishes || r0 + 16 * out_tile + out_row >= rows) return;
    floatx4 v = *reinterpret_cast<const floatx4*>(&tiles[0][out_tile][quad][out_row * 4]);
#pragma unroll
    for (int k = 1; k < kWaves; ++k) v += *reinterpret_cast<const floatx4*>(&tiles[k][out_tile][quad][out_row * 4]);
    store_epilogue(g, at_out, col, ein, v);
}

// ---------------------------------------------------------------------------
// Longer sequences.  An LDS row is 32 floats (128 bytes) of one matrix row as
// eight 16-byte chunks, chunk c at slot c ^ ((row >> 1) & 7): a direct load
// (global_load_lds, 64 lanes x 16 bytes side by side) applies the swizzle in
// the address each lane reads, and a fragment read's 16 rows fall into
// distinct banks.  The ring's buffers are separate __shared__ objects and the
// steps unrolled over them, so that the compiler adds no wait of its own for
// loads into another buffer.
// ---------------------------------------------------------------------------
constexpr int wait_imm(int vm) { return (vm & 15) | ((vm >> 4) << 14) | (7 << 4); }

template <int kLoads>
__device__ __forceinline__ void wait_and_sync() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(wait_imm(kLoads));
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

template <int kTM, int kTN, int kWM, int kWN, int kWK, int kStages>
__global__ __launch_bounds__(64 * kWM * kWN * kWK) void tile_kernel(ConvArgs g, int row_tiles, int panels, int slices) {
    constexpr int kBM = 16 * kTM * kWM, kBN = 16 * kTN * kWN;
    constexpr int kGroup = kWM * kWN;                 // waves of a K group
    constexpr int kLoads = (kBM + kBN) / 8 / kGroup;  // loads a wave issues per step, 8 rows each
    static_assert((kBM + kBN) % (8 * kGroup) == 0 && kStages >= 3 && kStages <= 4, "tile");
    constexpr int kPart = (kBM + kBN) * 32;  // floats a K group stages per step
    __shared__ __align__(16) float buffer0[kPart * kWK];
    __shared__ __align__(16) float buffer1[kPart * kWK];
    __shared__ __align__(16) float buffer2[kPart * kWK];
    __shared__ __align__(16) float buffer3[kStages > 3 ? kPart * kWK : 4];

    // Each XCD (block % 8) takes a contiguous eighth of the tiles in panel
    // order, so the row tiles that read one weight panel mostly share its L2.
    const int tiles = row_tiles * panels, share = (tiles + 7) >> 3;
    const int index = static_cast<int>(blockIdx.x & 7) * share + static_cast<int>(blockIdx.x >> 3);
    if (index >= tiles) return;  // the whole block
    const int panel = index / row_tiles, tile = index - panel * row_tiles;
    const int r0 = tile * kBM, n0 = panel * kBN;
    const int rows = g.m * g.streams.count;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wk = wave / kGroup, wg = wave % kGroup;
    const int m = lane & 15, group = lane >> 4;

    // this lane's source of load i: tile row 8 (wg + kGroup i) + lane / 8
    const float* source[kLoads];
    bool from_a[kLoads];  // wave-uniform: 8 rows are all activations or all weights
#pragma unroll
    for (int i = 0; i < kLoads; ++i) {
        const int row = 8 * (wg + kGroup * i) + (lane >> 3);
        const int chunk = (lane & 7) ^ ((row >> 1) & 7);
        from_a[i] = 8 * (wg + kGroup * i) < kBM;
        if (from_a[i]) {
            const Row at = locate(g, min(r0 + row, rows - 1));
            source[i] = g.a + at.delta + static_cast<size_t>(at.p) * g.channels_in + chunk * 4;
        } else {
            source[i] = g.w + static_cast<size_t>(min(n0 + row - kBM, g.n - 1)) * g.k + chunk * 4;
        }
    }
    // slice blockIdx.y of the parts (32 values of K each)
    const int first = (g.k >> 5) * static_cast<int>(blockIdx.y) / slices;
    const int parts = (g.k >> 5) * static_cast<int>(blockIdx.y + 1) / slices;
    const int steps = (parts - first + kWK - 1) / kWK;
    const ptrdiff_t tap_stride = static_cast<ptrdiff_t>(g.dilation) * g.channels_in;
    int part = first + wk;  // this K group's next part to load, and its (tap, channel)
    int tap = (32 * part) / g.channels_in, chan = 32 * part - tap * g.channels_in;
    auto buffer = [&](int stage) -> float* {
        return stage == 0 ? buffer0 : stage == 1 ? buffer1 : stage == 2 ? buffer2 : buffer3;
    };
    auto load = [&](int stage) {
        if (kWK == 1 || part < parts) {  // a last step may lack parts (the last steps wait for all loads)
            float* to = buffer(stage) + wk * kPart;
            const ptrdiff_t a_at = tap * tap_stride + chan, w_at = static_cast<ptrdiff_t>(part) * 32;
#pragma unroll
            for (int i = 0; i < kLoads; ++i)
                __builtin_amdgcn_global_load_lds((global_word*)(source[i] + (from_a[i] ? a_at : w_at)),
                                                 (lds_word*)(to + (wg + kGroup * i) * 256), 16, 0, 0);
        }
        part += kWK;
        chan += 32 * kWK;
        while (chan >= g.channels_in) chan -= g.channels_in, ++tap;
    };

    const int wm = (wg / kWN) * (16 * kTM), wn = (wg % kWN) * (16 * kTN);
    floatx4 acc[kTM][kTN];
#pragma unroll
    for (int i = 0; i < kTM; ++i)
#pragma unroll
        for (int j = 0; j < kTN; ++j) acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};
    // one tile a wave: the epilogue's operands are requested ahead of the loop
    constexpr bool kAhead = kTM * kTN == 1;
    EpilogueIn ein{};
    if (kAhead && slices == 1 && wk == 0) {
        const int r = min(r0 + wm + m, rows - 1), col = min(n0 + wn + 4 * group, g.n - 4);
        ein = load_epilogue(g, locate(g, r), col, col % g.channels_out);
    }
    // fragments: chunks 2 group and 2 group + 1 of a row
    const int slot0 = ((2 * group) ^ (m >> 1)) * 4, slot1 = ((2 * group + 1) ^ (m >> 1)) * 4;
    const int a_lane = wk * kPart + (wm + m) * 32, w_lane = wk * kPart + (kBM + wn + m) * 32;
    int at_part = first + wk;  // the part this wave multiplies next
    auto compute = [&](int stage) {
        if (kWK == 1 || at_part < parts) {
            const float* from = buffer(stage);
            floatx4 av[kTM][2], wv[kTN][2];
#pragma unroll
            for (int i = 0; i < kTM; ++i) {
                av[i][0] = load4(from + (a_lane + slot0) + 16 * i * 32);
                av[i][1] = load4(from + (a_lane + slot1) + 16 * i * 32);
            }
#pragma unroll
            for (int j = 0; j < kTN; ++j) {
                wv[j][0] = load4(from + (w_lane + slot0) + 16 * j * 32);
                wv[j][1] = load4(from + (w_lane + slot1) + 16 * j * 32);
            }
#pragma unroll
            for (int e = 0; e < 8; ++e)
#pragma unroll
                for (int i = 0; i < kTM; ++i)
#pragma unroll
                    for (int j = 0; j < kTN; ++j)
                        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(wv[j][e >> 2][e & 3], av[i][e >> 2][e & 3],
                                                                         acc[i][j], 0, 0, 0);
        }
        at_part += kWK;
    };

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

    if constexpr (kWK > 1) {  // the K groups' sums, added in group order
        float* sums = buffer0;  // [group - 1][wave][tile][lane] float4: at most the ring's first buffer
        static_assert((kWK - 1) * kGroup * kTM * kTN * 256 <= kPart * kWK, "partial tiles fit a buffer");
        __syncthreads();  // every wave is done with the ring
        if (wk > 0) {
#pragma unroll
            for (int i = 0; i < kTM; ++i)
#pragma unroll
                for (int j = 0; j < kTN; ++j)
                    *reinterpret_cast<floatx4*>(sums + ((((wk - 1) * kGroup + wg) * kTM + i) * kTN + j) * 256 + lane * 4) = acc[i][j];
        }
        __syncthreads();
        if (wk > 0) return;
#pragma unroll
        for (int k = 0; k < kWK - 1; ++k)
#pragma unroll
            for (int i = 0; i < kTM; ++i)
#pragma unroll
                for (int j = 0; j < kTN; ++j)
                    acc[i][j] += load4(sums + (((k * kGroup + wg) * kTM + i) * kTN + j) * 256 + lane * 4);
    }
    // acc[i][j] of lane (group, m): columns n0 + wn + 16 j + 4 group .. + 3 of row wm + 16 i + m
#pragma unroll
    for (int i = 0; i < kTM; ++i) {
        const int r = r0 + wm + 16 * i + m;
        if (r >= rows) continue;
        const Row at = locate(g, r);
#pragma unroll
        for (int j = 0; j < kTN; ++j) {
            const int col = n0 + wn + 16 * j + 4 * group;
            if (col >= g.n) continue;
            if (slices > 1)
                *reinterpret_cast<floatx4*>(g.partial + at.delta + (static_cast<size_t>(blockIdx.y) * g.m + at.p) * g.n + col) =
                    acc[i][j];
            else
                store_epilogue(g, at, col, kAhead ? ein : load_epilogue(g, at, col, col % g.channels_out), acc[i][j]);
        }
    }
}

// The slices' sums, added in slice order, and the epilogue: four columns a
// thread.
__global__ __launch_bounds__(64) void reduce_kernel(ConvArgs g, int slices) {
    const int quads = g.n >> 2, rows = g.m * g.streams.count;
    const int t = blockIdx.x * 64 + threadIdx.x;
    if (t >= rows * quads) return;
    const int r = t / quads, col = (t - r * quads) * 4;
    const Row at = locate(g, r);
    const EpilogueIn e = load_epilogue(g, at, col, col % g.channels_out);
    const size_t slice = static_cast<size_t>(g.m) * g.n;
    const float* p = g.partial + at.delta + static_cast<size_t>(at.p) * g.n + col;
    floatx4 sum = load4(p);
    for (int z0 = 1; z0 < slices; z0 += 4) {  // four slices' loads in flight
        floatx4 v[4];
#pragma unroll
        for (int d = 0; d < 4; ++d) v[d] = load4(p + min(z0 + d, slices - 1) * slice);
#pragma unroll
        for (int d = 0; d < 4; ++d)
            if (z0 + d < slices) sum += v[d];
    }
    store_epilogue(g, at, col, e, sum);
}

template <int kTM, int kTN, int kWM, int kWN, int kWK, int kStages>
hipError_t launch_tile(const ConvArgs& g, hipStream_t stream, int slices = 1) {
    constexpr int kBM = 16 * kTM * kWM, kBN = 16 * kTN * kWN;
    const int row_tiles = (g.m * g.streams.count + kBM - 1) / kBM, panels = (g.n + kBN - 1) / kBN;
    const unsigned blocks = (row_tiles * panels + 7) / 8 * 8;
    tile_kernel<kTM, kTN, kWM, kWN, kWK, kStages>
        <<<dim3(blocks, slices), 64 * kWM * kWN * kWK, 0, stream>>>(g, row_tiles, panels, slices);
    hipError_t st = hipGetLastError();
    if (st == hipSuccess && slices > 1) {
        reduce_kernel<<<(g.m * g.streams.count * (g.n / 4) + 63) / 64, 64, 0, stream>>>(g, slices);
        st = hipGetLastError();
    }
    return st;
}

template <int kTM, int kWaves>
hipError_t launch_rows(const ConvArgs& g, hipStream_t stream) {
    const dim3 grid(g.n / 16, (g.m * g.streams.count + 16 * kTM - 1) / (16 * kTM));
    rows_kernel<kTM, kWaves><<<grid, 64 * kWaves, 0, stream>>>(g);
    return hipGetLastError();
}

// How a product is summed, from one stream's rows and the layer's sizes alone.
// 16 x 16 tiles of one stream times `pieces` of K give the matrix cores their
// waves; residues of a block (tile_kernel) times K slices summed by a second
// launch.  Measured (us, weights from memory; 1 / 4 frames):
//   1024 x 4096, 4 / 16 rows: 16 pieces 9.7 / 9.9 (one slice 14.4 / 18)
//   1536 x 7168, 4 / 16 rows: 16 pieces 13.8 / 14.6 (one slice 24 / 28)
//   768 x 5376, 32 / 128 rows: 16 pieces 12.3, 8 pieces 20.3 (4: 24 / 25)
//   384 x 2688, 160 / 640 rows: 8 pieces 12.5, 2 pieces 23 (1: 30; 4 pieces
//     20.7, but 112 for six streams, where 2 allow 64 x 96 tiles, 82)
//   192 x 1344, 640 / 2560 rows: 4 pieces 8.8, 2 pieces 20 (1: 16 / 20.5)
//   96 x 672, 1920 / 7680 rows: 2 pieces 8.2, 1 piece 15.7 (1: 9.3; 2: 16.7)
struct Summation {
    bool rows;  // rows_kernel
    int residues, slices;
};
Summation summation(int m, int n, int k) {
    if (m <= 32 && k <= 1536) return {true, 16, 1};
    const int tiles = ((m + 15) / 16) * (n / 16);
    int pieces = tiles >= 2500 ? 1 : tiles >= 600 ? 2 : tiles >= 400 ? 4 : tiles >= 200 ? 8 : 16;
    while (pieces > 1 && pieces * 3 > k / 32) pieces >>= 1;  // at least 96 of K a piece
    return {false, pieces == 4 ? 4 : std::min(pieces, 2), pieces > 4 ? pieces / 2 : 1};
}

template <int kResidues>
hipError_t launch_tiles(const ConvArgs& g, int slices, hipStream_t stream) {
    // The tile's shape does not change a sum.  By the launch's size: 64 x 96
    // (32 x 96 for one residue, whose blocks are many) once that fills the CUs
    // several times (six streams, 3840 x 384 x 2688: 82 us, 32 x 32 98; 15360 x
    // 288 x 384: 45 us, 77), 16 x 32 for few rows or few tiles, else 32 x 32.
    const int rows = g.m * g.streams.count;
    const int tiles = ((rows + 15) / 16) * (g.n / 16);
    if constexpr (kResidues == 1) {
        if (g.n % 96 == 0 && tiles >= 8000) return launch_tile<1, 3, 2, 2, 1, 3>(g, stream, slices);
        return launch_tile<1, 1, 2, 2, 1, 4>(g, stream, slices);
    } else if constexpr (kResidues == 2) {
        if (rows <= 16) return launch_tile<1, 1, 1, 2, 2, 4>(g, stream, slices);
        if (g.n % 96 == 0 && tiles >= 5000) return launch_tile<2, 3, 2, 2, 2, 3>(g, stream, slices);
        return launch_tile<1, 1, 2, 2, 2, 4>(g, stream, slices);
    } else {
        if (tiles < 900) return launch_tile<1, 1, 1, 2, 4, 4>(g, stream, slices);
        return launch_tile<1, 1, 2, 2, 4, 3>(g, stream, slices);
    }
}

bool valid(const ConvArgs& g) {
    return g.a && g.w && g.m >= 1 && g.n >= 16 && g.n % 16 == 0 && g.k >= 32 && g.k % 32 == 0 && g.channels_in >= 32 &&
           g.channels_in % 32 == 0 && g.channels_out >= 4 && g.channels_out % 4 == 0 && g.dilation >= 1 &&
           g.streams.count >= 1 && g.streams.count <= kMaxStreams && (g.out || g.snake_out);
}

}  // namespace

size_t conv_partial_floats(int m, int n, int k) {
    const Summation how = summation(m, n, k);
    return how.slices > 1 ? static_cast<size_t>(how.slices) * m * n : 0;
}

hipError_t launch_conv(const ConvArgs& g, hipStream_t stream) {
    if (!valid(g)) return hipErrorInvalidValue;
    const Summation how = summation(g.m, g.n, g.k);
    if (how.rows) {
        // one tile of 16 rows a block while the blocks are few, else three
        // that share the weights' loads
        return g.m * g.streams.count <= 32 ? launch_rows<1, 16>(g, stream) : launch_rows<3, 16>(g, stream);
    }
    if (how.slices > 1 && !g.partial) return hipErrorInvalidValue;
    switch (how.residues) {
        case 1: return launch_tiles<1>(g, how.slices, stream);
        case 2: return launch_tiles<2>(g, how.slices, stream);
        default: return launch_tiles<4>(g, how.slices, stream);
    }
}

}  // namespace q3c
